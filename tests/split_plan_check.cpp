// CPU check of the split-KV plans (flash-mlm_amd/csrc/fmlm_split_plan.h): for many packed
// calls and scratch sizes, the records, groups and units of the plan that schedule_kernel
// makes stay within what the launch has room for.  Prints the plans that do not; exit
// status 1 if there are any.
#define __host__
#define __device__
#include "../flash-mlm_amd/csrc/fmlm_split_plan.h"

#include <cstdio>
#include <random>
#include <vector>

using namespace fmlm;

static int failures = 0, split_plans = 0, unsplit_plans = 0;

// H heads, sequences of len[b] tokens over keys[b] keys; slots workgroups at once; records
// of bq rows x D columns, rec_cap of them at most, in `scratch` bytes (0: as many as wanted)
static void check(const char* name, bool hpack, int H, const std::vector<int>& len, const std::vector<int>& keys, int D,
                  int bq, int slots, int rec_cap, int64_t scratch) {
  const int B = (int)len.size();
  fmlm_attn_params p{};
  p.B = B;
  p.H = H;
  p.D = D;
  for (int n : len) p.total_q += n;
  SplitCfg sc;
  sc.slots = slots;
  sc.rec_cap = rec_cap;
  sc.rec_bytes = ((int64_t)bq * (D * 4 + 8) + 15) / 16 * 16;
  if (scratch > 0 && !fit_records(p, bq, hpack, scratch, sc)) return;
  const SchedLayout l = sched_layout(p, bq, sc, hpack);

  // schedule_kernel's decision
  std::vector<int> tiles(B);
  std::vector<float> work(B);
  float units = 0.f, total = 0.f;
  int kmax = 0;
  for (int b = 0; b < B; ++b) {
    tiles[b] = ((hpack ? H : 1) * len[b] + bq - 1) / bq;
    work[b] = (float)((keys[b] + 63) / 64);
    units += (float)tiles[b] * (hpack ? 1 : H);
    total += (float)tiles[b] * (hpack ? 1 : H) * work[b];
    if (tiles[b] > 0) kmax = std::max(kmax, (int)work[b]);
  }
  int chunk = 0;
  if (sc.rec_cap > 0 && units < kSplitRounds * slots) {
    if (hpack) {
      float best = INFINITY;
      for (int S = 1; S <= 64; ++S) best = std::min(best, hpack_price(tiles.data(), work.data(), B, kmax, S, slots, sc.rec_cap).cost);
      for (int S = 1; S <= 64; ++S)
        chunk = std::max(chunk, hpack_take(hpack_price(tiles.data(), work.data(), B, kmax, S, slots, sc.rec_cap), best, kmax));
    } else {
      chunk = seq_chunk(tiles.data(), work.data(), B, H, total, slots, sc.rec_cap);
    }
  }
  int64_t n_units = 0, records = 0, groups = 0;
  for (int b = 0; b < B; ++b) {
    const int S = chunk > 0 ? split_parts(work[b], chunk) : 1;
    const int64_t t = (int64_t)tiles[b] * (hpack ? 1 : H);
    n_units += t * S;
    if (S > 1) groups += t;
    // head-packed parts may be numbered by their place in the call, unsplit tiles included
    if (S > 1 || (hpack && chunk > 0)) records += t * S;
  }
  (chunk > 0 ? split_plans : unsplit_plans)++;
  const bool ok = records <= sc.rec_cap && groups <= sc.rec_cap && n_units <= l.cap &&
                  (scratch == 0 || l.records_off + records * sc.rec_bytes <= scratch);
  if (!ok && failures++ < 10)
    std::printf("%s: H %d B %d tokens %d: %lld units of %lld, %lld records of %d, %lld groups, %lld bytes of %lld\n",
                name, H, B, p.total_q, (long long)n_units, (long long)l.cap, (long long)records, sc.rec_cap,
                (long long)groups, (long long)(l.records_off + records * sc.rec_bytes), (long long)scratch);
}

// the record count and tile rows of the 512-wide latent's launches on 256 slots
static void latent(const char* name, int H, const std::vector<int>& len, const std::vector<int>& keys, int64_t scratch) {
  int64_t rows = 0;
  for (int n : len) rows += (int64_t)H * n;
  const int bq = rows <= 4096 ? 64 : 128;
  const int rec_cap = ((rows + bq - 1) / bq + (int64_t)len.size() <= 256 ? 1 : 2) * 256;
  check(name, true, H, len, keys, 512, bq, 256, rec_cap, scratch);
}

int main() {
  const int64_t scratch = FMLM_NOALLOC_SCRATCH_BYTES;
  // more unsplit tiles than records in the library's scratch array
  latent("64 heads, 16 x 8 tokens, 4000 keys", 64, std::vector<int>(16, 8), std::vector<int>(16, 4000), scratch);
  latent("16 heads, 160 x 1 token, 2000 keys", 16, std::vector<int>(160, 1), std::vector<int>(160, 2000), scratch);
  latent("16 heads, 200 x 1 token, 2500 keys", 16, std::vector<int>(200, 1), std::vector<int>(200, 2500), scratch);
  latent("all empty", 16, {0, 0}, {0, 0}, scratch);

  // a few tokens in a long padded sequence: the tiles are those of the tokens
  for (int bq : {64, 128}) {
    fmlm_attn_params p{};
    p.B = 1;
    p.H = 64;
    p.N = 70000;
    p.total_q = 40;
    const bool ok = units_encodable(p, bq, queue_cap(p, bq, SplitCfg{}, true), true);
    p.total_q = p.N = 200000;
    const bool too_many = units_encodable(p, bq, queue_cap(p, bq, SplitCfg{}, true), true);
    if (!ok || too_many) {
      failures++;
      std::printf("units_encodable, %d rows per tile: %d for 40 tokens, %d for 200000\n", bq, ok, too_many);
    }
  }

  std::mt19937 gen(1);
  auto uni = [&](int lo, int hi) { return std::uniform_int_distribution<int>(lo, hi)(gen); };
  auto size = [&](int lo, int hi) {  // spread over the logarithm
    return (int)std::lround(std::exp(std::uniform_real_distribution<double>(std::log((double)lo), std::log((double)hi))(gen)));
  };
  for (int i = 0; i < 60000; ++i) {
    const int B = size(1, 300);
    std::vector<int> len(B), keys(B);
    const int most = size(1, 300), longest = size(1, 20000);
    for (int b = 0; b < B; ++b) {
      len[b] = uni(0, most);
      keys[b] = uni(0, 3) == 0 ? uni(0, longest) : longest;
    }
    const int H = uni(0, 1) ? 1 << uni(0, 7) : uni(1, 100);
    latent("latent", H, len, keys, uni(0, 1) ? scratch : size(1 << 16, 1 << 25));
    latent("latent", H, len, keys, 0);
    const int D = 16 << uni(0, 5), slots = 256 * uni(1, 4);
    check("latent, any record count", true, H, len, keys, D, uni(0, 1) ? 64 : 128, slots, uni(0, 1) ? uni(0, 2 * slots) : slots,
          size(1 << 16, 1 << 26));
    check("heads", false, H, len, keys, D, 16 << uni(0, 3), slots, 3 * slots, uni(0, 1) ? scratch : 0);
  }
  std::printf("%d plans split, %d not, %d wrong\n", split_plans, unsplit_plans, failures);
  return failures || split_plans < 1000 || unsplit_plans < 1000;
}
