"""GPU tests of key ranges split over workgroups and merged (dense calls with few query
tiles, the 512-wide latent with few query rows), against the float64 oracle and against
the same call unsplit.

Tolerance: 1e-2 as for every 16-bit forward test; the merged row differs from the unsplit
one by the rounding of its fp32 weights only, so the two are within one rounding of the
output type of each other (2^-8 relative at bf16, 2^-11 at fp16), plus 1e-5 for fp32."""

from __future__ import annotations

import ctypes
import random

import numpy as np
import pytest
import torch

from flash_mlm import InferenceCache, _lib, build_pack_metadata, flash_attn_mlm, flash_attn_mlm_compressed, \
    unpack_from_kernel
from flash_mlm.host import host as hh
from oracle import attention_ref as ar

pytestmark = pytest.mark.gpu


def _np(t):
    return t.detach().float().cpu().numpy().astype(np.float64)


def _randn(gen, shape, dtype, device, std=1.0):
    return (torch.randn(shape, generator=gen) * std).to(dtype).to(device)


DENSE = [
    # B, H, N, D, context rows, context batches, dtype: part counts that divide the key
    # tiles unevenly, one query row, a row past a tile, one row short of a key tile
    (1, 4, 1, 64, 2047, 1, torch.bfloat16),
    (2, 3, 65, 64, 2500, 2, torch.float16),
    (1, 2, 17, 128, 6001, 1, torch.bfloat16),
    (1, 1, 128, 256, 1300, 1, torch.float16),
    (3, 2, 130, 32, 2049, 3, torch.bfloat16),
    (1, 3, 600, 16, 3001, 1, torch.float16),
    (1, 2, 33, 64, 2050, 1, torch.float32),
]


@pytest.mark.parametrize("B,H,N,D,C,cbs,dtype", DENSE)
def test_dense_split_matches_oracle_and_unsplit(B, H, N, D, C, cbs, dtype, device):
    gen = torch.Generator().manual_seed(D + N)
    q, k, v = (_randn(gen, (B, H, N, D), dtype, device) for _ in range(3))
    kc, vc = (_randn(gen, (cbs * H * C, D), dtype, device) for _ in range(2))
    cache = InferenceCache()
    cache.prefill_kv_cache(0, k_cache=kc, v_cache=vc, context_batch_size=cbs, is_mla=False, num_heads=H, head_dim=D)
    scale = D ** -0.5
    out, plan = hh._dense_impl(q, k, v, scale, cache, 0, False, None, False, run=False)
    assert plan.records > 0, "the shape is meant to split"
    plan()
    tol = 1e-5 if dtype == torch.float32 else 1e-2
    ref = ar.mlm_attention_dense(_np(q), _np(k), _np(v), scale, k_cache=_np(kc), v_cache=_np(vc), context_len=C,
                                 context_batch_size=cbs)
    np.testing.assert_allclose(_np(out), ref, atol=tol, rtol=tol)
    again = flash_attn_mlm(q, k, v, scale, inference_cache=cache, layer_id=0)
    assert torch.equal(again, out)
    # without a workspace the C ABI runs the call unsplit
    p = _lib.AttnParams.from_buffer_copy(plan.params)
    whole = torch.full_like(out, float("nan"))
    p.o, p.workspace, p.workspace_bytes = whole.data_ptr(), None, 0
    _lib.check(plan.lib.fmlm_attn_fwd(ctypes.byref(p), plan.stream), "fmlm_attn_fwd")
    ulp = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11, torch.float32: 1e-5}[dtype]
    torch.testing.assert_close(out.float(), whole.float(), atol=ulp * float(whole.float().abs().max()), rtol=ulp)


def _split_groups(meta):
    """Split groups of the one schedule of a metadata (header word 1)."""
    (sched,) = meta.kernel_schedules.values()
    return int(sched[:8].view(torch.int32)[1])


@pytest.mark.parametrize("B,H,N,C,cbs", [(1, 4, 20, 3000, 1), (2, 3, 130, 2050, 2), (1, 1, 1, 1500, 1)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_dense_latent_split_matches_oracle_and_unsplit(dtype, B, H, N, C, cbs, device):
    """The 512-wide latent in a dense call (per-head main keys, one latent context): tiles of
    128 rows of one head, cut and merged."""
    gen = torch.Generator().manual_seed(N)
    D = 512
    q, k = (_randn(gen, (B, H, N, D), dtype, device, 0.5) for _ in range(2))
    kc = _randn(gen, (cbs * C, D), dtype, device, 0.5)
    cache = InferenceCache()
    cache.prefill_kv_cache(0, k_cache=kc, context_batch_size=cbs, is_mla=True, num_heads=H, head_dim=D)
    scale = D ** -0.5
    out, plan = hh._dense_impl(q, k, k, scale, cache, 0, True, None, False, run=False)
    assert plan.records > 0, "the shape is meant to split"
    plan()
    ref = ar.mlm_attention_dense(_np(q), _np(k), _np(k), scale, is_mla=True, k_cache=_np(kc), context_len=C,
                                 context_batch_size=cbs)
    np.testing.assert_allclose(_np(out), ref, atol=1e-2, rtol=1e-2)
    p = _lib.AttnParams.from_buffer_copy(plan.params)
    whole = torch.full_like(out, float("nan"))
    p.o, p.workspace, p.workspace_bytes = whole.data_ptr(), None, 0
    _lib.check(plan.lib.fmlm_attn_fwd(ctypes.byref(p), plan.stream), "fmlm_attn_fwd")
    # P is rounded to 16 bits against each part's own maximum: two roundings of weights and
    # one of the output apart
    ulp = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}[dtype]
    torch.testing.assert_close(out.float(), whole.float(), atol=2 * ulp * float(whole.float().abs().max()), rtol=ulp)


@pytest.mark.parametrize("H,lengths,ctx", [
    # one tile of 64 rows, by work all 16 parts on one XCD
    (16, [3], [4097]),
    # by work the fullest XCD has 33 (38) parts, its 32 CUs take one each
    (64, [8] * 16, random.Random(0).choices(range(2000, 6001), k=16)),
    (64, [8] * 16, sorted(random.Random(2).choices(range(2000, 6001), k=16))),
])
def test_latent_parts_are_dealt_by_count(H, lengths, ctx, device):
    """Where parts placed by work would crowd an XCD, the queues get equal counts instead;
    every (tile, part) is one unit, and every part has a record of its own."""
    gen = torch.Generator().manual_seed(H)
    dtype, D, N, B = torch.bfloat16, 512, max(lengths), len(lengths)
    q, k = (_randn(gen, (B, H, N, D), dtype, device, 0.5) for _ in range(2))
    cu = [0, *np.cumsum(ctx).tolist()]
    kc = _randn(gen, (cu[-1], D), dtype, device, 0.5)
    cache = InferenceCache()
    cache.prefill_kv_cache(0, k_cache=kc, total_context_len=cu[-1], context_batch_size=B, is_mla=True, num_heads=H,
                           cu_seqlens_kv=torch.tensor(cu, dtype=torch.int32, device=device), head_dim=D)
    meta = build_pack_metadata(torch.tensor(lengths, dtype=torch.int32, device=device), N, 64)
    out = flash_attn_mlm_compressed(q, k, k, H, meta, D ** -0.5, cache, 0, is_mla=True, block_n=64)
    (sched,) = meta.kernel_schedules.values()
    words = sched.cpu().numpy().view(np.int32)
    cap, queues = int(words[5]), words[8:16]
    assert _split_groups(meta) > 0
    assert queues.max() - queues.min() <= 1 and queues.sum() == words[0]
    units = words[64:64 + 8 * cap * 4].reshape(8, cap, 4)
    seen, records = set(), set()
    for x in range(8):
        for b, ht, rec0, w in units[x, :queues[x]]:
            part, parts = ((int(w) >> 20) & 31, ((int(w) >> 25) & 31) + 1) if w >= 0 else (0, 1)
            seen.add((int(b), int(ht) >> 16, part))
            if parts > 1:
                records.add(int(rec0) + part)
    bq = 64 if H * sum(lengths) <= 4096 else 128
    tiles = sum(-(-H * n // bq) for n in lengths)
    assert len(seen) == words[0] and len({t[:2] for t in seen}) == tiles
    assert len(records) == sum(1 for _ in seen) and max(records) < words[0]
    ref = ar.mlm_attention_packed(_np(q), _np(k), _np(k), lengths, D ** -0.5, is_mla=True, k_cache=_np(kc),
                                  cu_seqlens_kv=cu, total_context_len=cu[-1], context_batch_size=B)
    np.testing.assert_allclose(_np(unpack_from_kernel(out, meta, H)), ref, atol=1e-2, rtol=1e-2)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("H,lengths,ctx", [
    (64, [1, 0, 4, 2], [2000, 900, 0, 5]),       # tiles of 64, 128 and 256 rows, short and empty contexts
    (16, [3], [4097]),                           # one tile, the most parts
    (5, [7, 1, 30], [333, 1024, 64 * 9]),        # odd heads: rows of a tile span heads
    (32, [4, 3] * 40, [640, 517] * 40),          # many groups: the merge takes larger chunks
])
def test_latent_split_matches_oracle(H, lengths, ctx, paged, dtype, device):
    gen = torch.Generator().manual_seed(H)
    D, N, B = 512, max(lengths), len(lengths)
    q, k = (_randn(gen, (B, H, N, D), dtype, device, 0.5) for _ in range(2))
    cu = [0, *np.cumsum(ctx).tolist()]
    kc = _randn(gen, (cu[-1], D), dtype, device, 0.5)
    cache = InferenceCache()
    if paged:
        need = [(c + 63) // 64 for c in ctx]
        pool = torch.zeros((1, sum(need), 64, D), dtype=dtype, device=device)
        table = torch.zeros((B, max(need)), dtype=torch.int32)
        for b, c in enumerate(ctx):
            first = sum(need[:b])
            table[b, :need[b]] = torch.arange(first, first + need[b], dtype=torch.int32)
            pool[0, first:first + need[b]].view(-1, D)[:c] = kc[cu[b]:cu[b + 1]]
        cache.prefill_paged_kv_cache(0, k_pages=pool, block_table=table.to(device),
                                     context_lens=torch.tensor(ctx, dtype=torch.int32), is_mla=True, num_heads=H,
                                     head_dim=D)
    else:
        cache.prefill_kv_cache(0, k_cache=kc, total_context_len=cu[-1], context_batch_size=B, is_mla=True,
                               cu_seqlens_kv=torch.tensor(cu, dtype=torch.int32, device=device), num_heads=H,
                               head_dim=D)
    meta = build_pack_metadata(torch.tensor(lengths, dtype=torch.int32, device=device), N, 64)
    scale = D ** -0.5
    out = flash_attn_mlm_compressed(q, k, k, H, meta, scale, cache, 0, is_mla=True, block_n=64)
    assert _split_groups(meta) > 0, "the shape is meant to split"
    ref = ar.mlm_attention_packed(_np(q), _np(k), _np(k), lengths, scale, is_mla=True, k_cache=_np(kc),
                                  cu_seqlens_kv=cu, total_context_len=cu[-1], context_batch_size=B)
    np.testing.assert_allclose(_np(unpack_from_kernel(out, meta, H)), ref, atol=1e-2, rtol=1e-2)


def test_split_launches_of_one_schedule_do_not_share_partial_results(device):
    """Calls on the same metadata from two streams may overlap: each brings its own records."""
    gen = torch.Generator().manual_seed(9)
    B, H, N, D = 4, 32, 4, 512
    meta = build_pack_metadata(torch.tensor([4, 1, 3, 2], dtype=torch.int32, device=device), N, 64)
    cases = []
    for _ in range(2):
        q, k = (_randn(gen, (B, H, N, D), torch.bfloat16, device, 0.5) for _ in range(2))
        kc = _randn(gen, (B * 1500, D), torch.bfloat16, device, 0.5)
        cache = InferenceCache()
        cache.prefill_kv_cache(0, k_cache=kc, total_context_len=B * 1500, context_batch_size=B, is_mla=True,
                               cu_seqlens_kv=torch.arange(B + 1, dtype=torch.int32, device=device) * 1500,
                               num_heads=H, head_dim=D)
        cases.append((q, k, cache))

    def call(c):
        return flash_attn_mlm_compressed(c[0], c[1], c[1], H, meta, D ** -0.5, c[2], 0, is_mla=True, block_n=64)

    want = [call(c) for c in cases]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    got = [[], []]
    for _ in range(20):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                got[i].append(call(cases[i]))
    torch.cuda.synchronize()
    for i in range(2):
        for g in got[i]:
            assert torch.equal(g, want[i])


@pytest.mark.parametrize("way", ["dense", "latent"])
def test_split_call_in_a_graph(way, device):
    """A captured call that splits (its records come from the graph's own memory) replays to
    the eager result, with other calls between the replays."""
    gen = torch.Generator().manual_seed(12)
    cache, dtype = InferenceCache(), torch.bfloat16
    if way == "dense":
        H, D, C = 2, 128, 3000
        q, k, v = (_randn(gen, (1, H, 20, D), dtype, device) for _ in range(3))
        kc, vc = (_randn(gen, (H * C, D), dtype, device) for _ in range(2))
        cache.prefill_kv_cache(0, k_cache=kc, v_cache=vc, context_batch_size=1, is_mla=False, num_heads=H, head_dim=D)

        def call():
            return flash_attn_mlm(q, k, v, 0.1, inference_cache=cache, layer_id=0)
    else:
        B, H, D, C = 2, 16, 512, 1500
        q, k = (_randn(gen, (B, H, 3, D), dtype, device, 0.5) for _ in range(2))
        kc = _randn(gen, (B * C, D), dtype, device, 0.5)
        cu = torch.arange(B + 1, dtype=torch.int32, device=device) * C
        cache.prefill_kv_cache(0, k_cache=kc, total_context_len=B * C, cu_seqlens_kv=cu, context_batch_size=B,
                               is_mla=True, num_heads=H, head_dim=D)
        meta = build_pack_metadata(torch.tensor([3, 1], dtype=torch.int32, device=device), 3, 64)

        def call():
            return flash_attn_mlm_compressed(q, k, k, H, meta, 0.05, cache, 0, is_mla=True, block_n=64)

    want = call()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    for _ in range(4):
        out.zero_()
        graph.replay()
        eager = call()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(eager, want)


@pytest.mark.parametrize("D,H,mla", [(64, 4, False), (512, 16, True)])
def test_schedule_holds_the_records_or_each_call_brings_them(D, H, mla, device):
    """A schedule without room for the split records is only built, and only run, with
    FMLM_FLAG_OWN_RECORDS and a workspace for them; without the flag the records are in the
    schedule buffer, also when the caller passes that buffer as the workspace too."""
    gen = torch.Generator().manual_seed(21)
    dtype, lengths, C = torch.bfloat16, [3, 2], 3000
    N, B = max(lengths), len(lengths)
    q, k, v = (_randn(gen, (B, H, N, D), dtype, device, 0.5) for _ in range(3))
    hk = 1 if mla else H
    kc, vc = _randn(gen, (hk * B * C, D), dtype, device, 0.5), None if mla else _randn(gen, (hk * B * C, D), dtype, device, 0.5)
    cache = InferenceCache()
    cache.prefill_kv_cache(0, k_cache=kc, v_cache=vc, total_context_len=B * C, context_batch_size=B, is_mla=mla,
                           cu_seqlens_kv=torch.arange(B + 1, dtype=torch.int32, device=device) * C, num_heads=H,
                           head_dim=D)
    meta = build_pack_metadata(torch.tensor(lengths, dtype=torch.int32, device=device), N, 64)
    want, plan = hh._compressed_impl(q, k, v, H, meta, D ** -0.5, cache, 0, mla, None, 64, 64, False, False, False,
                                     run=False)
    assert plan.records > 0, "the shape is meant to split"
    plan()
    lib, stream, e_workspace = plan.lib, plan.stream, -5
    out = torch.full_like(want, float("nan"))

    def block():
        p = _lib.AttnParams.from_buffer_copy(plan.params)
        p.o, p.workspace, p.workspace_bytes = out.data_ptr(), None, 0
        return p

    p = block()
    assert p.flags & _lib.FLAG_OWN_RECORDS
    assert lib.fmlm_attn_fwd(ctypes.byref(p), stream) == e_workspace
    p = block()
    p.flags &= ~_lib.FLAG_OWN_RECORDS
    p.schedule = None
    nbytes, records = lib.fmlm_attn_workspace_bytes(ctypes.byref(p)), lib.fmlm_attn_records_bytes(ctypes.byref(p))
    assert records == plan.records
    buf = torch.empty(nbytes, dtype=torch.uint8, device=device)
    assert lib.fmlm_attn_schedule(ctypes.byref(p), buf.data_ptr(), nbytes - 1, stream) == e_workspace
    assert lib.fmlm_attn_schedule(ctypes.byref(p), buf.data_ptr(), nbytes, stream) == 0
    p.schedule = p.workspace = buf.data_ptr()
    p.workspace_bytes = nbytes
    for _ in range(2):  # the first run leaves the schedule as it was
        out.fill_(float("nan"))
        assert lib.fmlm_attn_fwd(ctypes.byref(p), stream) == 0
        torch.cuda.synchronize()
        assert torch.equal(out, want)


@pytest.mark.parametrize("plan_on_side", [True, False])
def test_records_of_a_run_from_another_stream(plan_on_side, device):
    """A prepared launch keeps its stream: the records of a run started while another
    stream is current are that stream's memory, which a new tensor of the current stream
    never gets while the launch may still be running."""
    gen = torch.Generator().manual_seed(3)
    H, D, C = 2, 64, 4000
    q, k, v = (_randn(gen, (1, H, 9, D), torch.bfloat16, device) for _ in range(3))
    kc, vc = (_randn(gen, (H * C, D), torch.bfloat16, device) for _ in range(2))
    cache = InferenceCache()
    cache.prefill_kv_cache(0, k_cache=kc, v_cache=vc, context_batch_size=1, is_mla=False, num_heads=H, head_dim=D)
    want = flash_attn_mlm(q, k, v, 0.125, inference_cache=cache, layer_id=0)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    own, other = (side, torch.cuda.current_stream()) if plan_on_side else (torch.cuda.current_stream(), side)
    with torch.cuda.stream(own):
        out, plan = hh._dense_impl(q, k, v, 0.125, cache, 0, False, None, False, run=False)
    assert plan.records > 0 and plan.stream == own.cuda_stream
    used = set()
    with torch.cuda.stream(other):
        for _ in range(3):
            plan()
            used.add(plan.params.workspace)
        fresh = [torch.empty(plan.records, dtype=torch.uint8, device=device) for _ in range(4)]
    assert used.isdisjoint(t.data_ptr() for t in fresh)
    torch.cuda.synchronize()
    assert torch.equal(out, want)
