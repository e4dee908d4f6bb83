// Split-KV sizing: how many records a launch may use and how long the parts of its key
// ranges are.  Plain C++ (no HIP types), used by the host, by schedule_kernel and by a CPU
// test that checks that no plan has more parts than records or more units than workgroups.
#pragma once

#include <stdint.h>

#include <algorithm>
#include <cmath>

#include "../../include/flash_mlm_hip.h"

namespace fmlm {

constexpr int kXcds = 8;
constexpr int kMaxSplits = 16;
constexpr int kMinSplitTiles = 8;   // key tiles per part at least
constexpr float kSplitRounds = 1.5f;
constexpr int kMinHpackTiles = 4;      // head-packed: key tiles per part at least
constexpr float kHpackPartCost = 4.f;  // and a part's start, end and merge, in key tiles

// Split-KV sizing: the GPU's workgroup slots for this kernel, the record capacity and
// the record size.
struct SplitCfg {
  int slots = 0;
  int rec_cap = 0;        // 0: no split
  int64_t rec_bytes = 0;  // per record: rows x (D fp32 + m + l)
  int dense_parts = 1;    // dense call: parts per query tile
};

// Parts of a key range of `work` tiles that is cut every `chunk` tiles.
__host__ __device__ inline int split_parts(float work, int chunk) {
  const float n = ceilf(work / (float)chunk);
  return n > kMaxSplits ? kMaxSplits : n > 1.f ? (int)n : 1;
}

// Part length of a call that is not head-packed, 0 when it is not split: about total /
// (kSplitRounds * slots) key tiles (total: query tiles x key tiles of the call), at least
// kMinSplitTiles, doubled until the records fit.
__host__ __device__ inline int seq_chunk(const int* tiles, const float* work, int B, int H, float total, int slots,
                                         int rec_cap) {
  int chunk = (int)ceilf(total / (kSplitRounds * slots));
  if (chunk < kMinSplitTiles) chunk = kMinSplitTiles;
  for (int it = 0; it < 24; ++it, chunk *= 2) {
    float recs = 0.f;
    for (int b = 0; b < B; ++b) {
      const int S = split_parts(work[b], chunk);
      if (S > 1) recs += (float)tiles[b] * H * S;
    }
    if (recs <= (float)rec_cap) return chunk;
  }
  return 0;
}

// Head-packed tiles fill a CU each (128 KiB of LDS), so parts run in whole rounds of
// `slots`.  The price of S parts for the longest sequence (kmax key tiles; the others'
// parts as long): rounds x (key tiles of a part + what a part costs besides).  Every tile
// of a call that is split takes a record per part, also one that is not cut itself, so a
// plan of more parts than records has an infinite price.
struct HpackPrice {
  float cost;
  int chunk;
};
__host__ __device__ inline HpackPrice hpack_price(const int* tiles, const float* work, int B, int kmax, int S,
                                                  int slots, int rec_cap) {
  HpackPrice r;
  r.chunk = (int)ceilf((float)kmax / (float)S);
  if (r.chunk < kMinHpackTiles) r.chunk = kMinHpackTiles;
  float parts = 0.f;
  for (int b = 0; b < B; ++b) parts += (float)tiles[b] * split_parts(work[b], r.chunk);
  r.cost = ceilf(parts / slots) * (r.chunk + kHpackPartCost);
  if (parts > (float)rec_cap || S > kMaxSplits) r.cost = INFINITY;
  return r;
}
// the part length that a price of `best`, the lowest of all, stands for; 0: no split, also
// when no plan fits the records (all prices are infinite)
__host__ __device__ inline int hpack_take(const HpackPrice& r, float best, int kmax) {
  return r.cost < INFINITY && r.cost == best && r.chunk < kmax ? r.chunk : 0;
}

// Units of an unsplit packed call, at most: sequence b has ceil(L_b / bq) <= L_b / bq + 1
// query tiles per head (head-packed: ceil(H L_b / bq) in all).
inline int64_t max_units(const fmlm_attn_params& p, int bq, bool hpack) {
  return hpack ? ((int64_t)p.H * p.total_q + bq - 1) / bq + p.B
               : (int64_t)p.H * (((int64_t)p.total_q + bq - 1) / bq + p.B);
}

// Entries per queue of a packed call: a bound on the launch's units, so that one queue
// can take all of them whatever the placement; with splits, which happen only below
// kSplitRounds * slots unsplit units, add every split part.
inline int64_t queue_cap(const fmlm_attn_params& p, int bq, const SplitCfg& sc, bool hpack) {
  int64_t units = max_units(p, bq, hpack);
  if (sc.rec_cap > 0) {
    const int64_t split_units = std::min(units, (int64_t)(kSplitRounds * sc.slots) + 1) + sc.rec_cap;
    units = split_units > units ? split_units : units;
  }
  return units;
}

// Schedule buffer layout (see schedule_kernel): header, 8 queues, groups, records.
struct SchedLayout {
  int64_t cap, units_off, groups_off, records_off, bytes;
};

inline SchedLayout sched_layout(const fmlm_attn_params& p, int bq, const SplitCfg& sc, bool hpack) {
  const int64_t entry = 16;  // int4
  SchedLayout l;
  l.cap = queue_cap(p, bq, sc, hpack);
  l.units_off = 256;
  l.groups_off = l.units_off + kXcds * l.cap * entry;
  l.groups_off = (l.groups_off + 255) / 256 * 256;
  l.records_off = l.groups_off + (int64_t)sc.rec_cap * entry;
  l.records_off = (l.records_off + 255) / 256 * 256;
  l.bytes = l.records_off + (int64_t)sc.rec_cap * sc.rec_bytes;
  return l;
}

// Whether the call's units fit their encoding: 16-bit heads, 16-bit tiles of a sequence's
// rows (head-packed: of its H times as many), 32-bit indices of queue entries.
inline bool units_encodable(const fmlm_attn_params& p, int bq, int64_t cap, bool hpack) {
  const int64_t most = p.N > 0 && p.N < p.total_q ? p.N : p.total_q;  // tokens of a sequence
  const int64_t rows = hpack ? (int64_t)p.H * most : p.N;
  return kXcds * cap <= 0x7fffffff && p.H <= 0xffff && (rows + bq - 1) / bq <= 0xffff;
}

// Cuts the record count of a packed call so that the schedule and the records fit `cap`
// bytes.  No split when fewer would fit than one per workgroup slot (head-packed: than the
// units the unsplit call can have, each of which takes a record, see hpack_price).  Returns
// false when even the unsplit schedule does not fit.
inline bool fit_records(const fmlm_attn_params& p, int bq, bool hpack, int64_t cap, SplitCfg& sc) {
  auto fits = [&](int rec_cap) {
    SplitCfg t = sc;
    t.rec_cap = rec_cap;
    return sched_layout(p, bq, t, hpack).bytes <= cap;
  };
  if (fits(sc.rec_cap)) return true;
  // the layout grows with the record count: the largest count in [lo, rec_cap) that fits
  int64_t lo = hpack ? max_units(p, bq, true) : sc.slots, hi = sc.rec_cap - 1;
  if (sc.rec_cap > 0 && lo <= hi && fits((int)lo)) {
    while (lo < hi) {
      const int64_t mid = lo + (hi - lo + 1) / 2;
      if (fits((int)mid))
        lo = mid;
      else
        hi = mid - 1;
    }
    sc.rec_cap = (int)lo;
    return true;
  }
  sc.rec_cap = 0;
  return fits(0);
}

}  // namespace fmlm
