"""GPU tests of the fp32 kernels (matrix cores) at the sizes where their tiles end, against
the float64 oracle on the same inputs.

Tolerance: a score is a sum of D products of values around 1 in fp32, off by up to about
sqrt(D) * 2^-24 * its size (at most 8 here), which is its weight's relative error; the
output, at most about 3, is then off by less than 16 * 8 * 6e-8 * 3 = 2.3e-5 at D = 256."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from flash_mlm import InferenceCache, build_pack_metadata, flash_attn_mlm, flash_attn_mlm_compressed, \
    unpack_from_kernel
from oracle import attention_ref as ar

pytestmark = pytest.mark.gpu
TOL = 2.5e-5


def _np(t):
    return t.detach().cpu().numpy().astype(np.float64)


def _case(device, D, H, lengths, ctx, seed, mla=False, grad=False):
    gen = torch.Generator().manual_seed(seed)
    B, N = len(lengths), max(lengths)
    r = lambda *shape: torch.randn(shape, generator=gen).to(device).requires_grad_(grad)  # noqa: E731
    q, k, v = (r(B, H, N, D) for _ in range(3))
    cu = [0, *np.cumsum(ctx).tolist()]
    hk = 1 if mla else H
    kc, vc = r(hk * cu[-1], D), None if mla else r(hk * cu[-1], D)
    cache = InferenceCache()
    cache.prefill_kv_cache(0, k_cache=kc, v_cache=vc, total_context_len=cu[-1], context_batch_size=len(ctx),
                           cu_seqlens_kv=torch.tensor(cu, dtype=torch.int32, device=device), is_mla=mla,
                           num_heads=H, head_dim=D)
    meta = build_pack_metadata(torch.tensor(lengths, dtype=torch.int32, device=device), N, 64)
    return q, k, v, kc, vc, cu, cache, meta


# sequence lengths around the 16- and 32-row query tiles and the 16- and 64-key tiles, with
# context lengths that leave none, some or all of a tile's waves without keys; (H, lengths,
# ctx) of the last case fill the chip with wide query tiles
EDGES = [
    (3, [1, 15, 16, 17, 33, 64, 65], [0, 1, 16, 63, 64, 65, 130]),
    (2, [31, 0, 5], [48]),
    (16, [200, 129, 256], [17, 300, 0]),
]


@pytest.mark.parametrize("causal,mla", [(False, False), (True, False), (False, True)])
@pytest.mark.parametrize("H,lengths,ctx", EDGES)
@pytest.mark.parametrize("D", [16, 32, 64, 128, 256])
def test_f32_forward_edges(D, H, lengths, ctx, causal, mla, device):
    q, k, v, kc, vc, cu, cache, meta = _case(device, D, H, lengths, ctx, D + H, mla)
    scale = D ** -0.5
    out = flash_attn_mlm_compressed(q, k, v, H, meta, scale, cache, 0, is_mla=mla, block_n=64,
                                    causal_query_seq_attn=causal)
    ref = ar.mlm_attention_packed(_np(q), _np(k), _np(k if mla else v), lengths, scale, is_mla=mla,
                                  causal_query_seq_attn=causal, k_cache=_np(kc),
                                  v_cache=None if mla else _np(vc), cu_seqlens_kv=cu, total_context_len=cu[-1],
                                  context_batch_size=len(ctx))
    np.testing.assert_allclose(_np(unpack_from_kernel(out, meta, H)), ref, atol=TOL, rtol=TOL)


@pytest.mark.parametrize("causal,mla", [(False, False), (True, False), (False, True)])
@pytest.mark.parametrize("H,lengths,ctx", EDGES)
@pytest.mark.parametrize("D", [16, 32, 64, 128, 256])
def test_f32_backward_edges(D, H, lengths, ctx, causal, mla, device):
    """Gradients within 2e-5 of the largest entry: dS = P (dP - delta) with P off by at most
    16 * 8 * 6e-8 = 8e-6 of itself (above) and dP - delta by about as much of its range."""
    q, k, v, kc, vc, cu, cache, meta = _case(device, D, H, lengths, ctx, D + H, mla, grad=True)
    scale = D ** -0.5
    out = flash_attn_mlm_compressed(q, k, v, H, meta, scale, cache, 0, is_mla=mla, block_n=64,
                                    causal_query_seq_attn=causal)
    dout = torch.randn(out.shape, generator=torch.Generator().manual_seed(1)).to(device)
    leaves = [q, k, kc] if mla else [q, k, v, kc, vc]
    got = torch.autograd.grad(out, leaves, dout)
    ref = ar.mlm_attention_packed_backward(
        _np(q), _np(k), _np(k if mla else v), _np(unpack_from_kernel(dout, meta, H)), lengths, scale, is_mla=mla,
        causal_query_seq_attn=causal, k_cache=_np(kc), v_cache=None if mla else _np(vc), cu_seqlens_kv=cu,
        total_context_len=cu[-1], context_batch_size=len(ctx))
    ref = [ref[0], ref[1], ref[3]] if mla else ref
    for name, g, r in zip(["q", "k", "kc"] if mla else ["q", "k", "v", "kc", "vc"], got, ref):
        worst = np.abs(_np(g) - r).max() / np.abs(r).max()
        assert worst <= 2e-5, (name, worst)


@pytest.mark.parametrize("D,mla", [(16, False), (64, False), (128, True), (256, False)])
def test_f32_packed_split(D, mla, device):
    """Few queries over long ragged contexts: the schedule splits key ranges, and the fp32
    records are merged; outputs, row statistics (through the backward) and gradients."""
    H, lengths, ctx = 2, [5, 0, 9], [6000, 300, 3001]
    q, k, v, kc, vc, cu, cache, meta = _case(device, D, H, lengths, ctx, D, mla, grad=True)
    scale = D ** -0.5
    out = flash_attn_mlm_compressed(q, k, v, H, meta, scale, cache, 0, is_mla=mla, block_n=64)
    (sched,) = meta.kernel_schedules.values()
    assert int(sched[:8].view(torch.int32)[1]) > 0, "the shape is meant to split"
    kw = dict(is_mla=mla, k_cache=_np(kc), v_cache=None if mla else _np(vc), cu_seqlens_kv=cu,
              total_context_len=cu[-1], context_batch_size=len(ctx))
    ref = ar.mlm_attention_packed(_np(q), _np(k), _np(k if mla else v), lengths, scale, **kw)
    np.testing.assert_allclose(_np(unpack_from_kernel(out.detach(), meta, H)), ref, atol=TOL, rtol=TOL)
    dout = torch.randn(out.shape, generator=torch.Generator().manual_seed(1)).to(device)
    leaves = [q, k, kc] if mla else [q, k, v, kc, vc]
    got = torch.autograd.grad(out, leaves, dout)
    want = ar.mlm_attention_packed_backward(_np(q), _np(k), _np(k if mla else v),
                                            _np(unpack_from_kernel(dout, meta, H)), lengths, scale, **kw)
    want = [want[0], want[1], want[3]] if mla else want
    for name, g, r in zip(["q", "k", "kc"] if mla else ["q", "k", "v", "kc", "vc"], got, want):
        worst = np.abs(_np(g) - r).max() / np.abs(r).max()
        assert worst <= 2e-5, (name, worst)


@pytest.mark.parametrize("D", [16, 64, 256])
def test_f32_infinity_in_a_last_value_row(D, device):
    """A value that is infinite in the last row of a key range reaches that column of every
    row that attends to it and nothing else: key slots past a range's end hold no copy of
    it (0 * inf would be NaN)."""
    H, lengths, ctx = 2, [5, 33, 16], [17, 3, 70]
    q, k, v, kc, vc, cu, cache, meta = _case(device, D, H, lengths, ctx, D)
    v[0, 1, lengths[0] - 1, 3] = float("inf")  # sequence 0, head 1: main keys
    vc[cu[2] - 1, 7] = float("-inf")           # sequence 1, head 0: context
    out = unpack_from_kernel(flash_attn_mlm_compressed(q, k, v, H, meta, D ** -0.5, cache, 0, block_n=64), meta, H)
    finite_v, finite_vc = v.clone(), vc.clone()
    finite_v[0, 1, lengths[0] - 1, 3] = finite_vc[cu[2] - 1, 7] = 0.0
    ref = ar.mlm_attention_packed(_np(q), _np(k), _np(finite_v), lengths, D ** -0.5, k_cache=_np(kc),
                                  v_cache=_np(finite_vc), cu_seqlens_kv=cu, total_context_len=cu[-1],
                                  context_batch_size=len(ctx))
    ref[0, 1, :lengths[0], 3] = np.inf
    ref[1, 0, :lengths[1], 7] = -np.inf
    np.testing.assert_allclose(_np(out), ref, atol=TOL, rtol=TOL)


@pytest.mark.parametrize("D", [16, 64, 256])
def test_f32_infinity_in_a_last_gradient_row(D, device):
    """The same for dO: one infinite entry in a sequence's last row makes that column of the
    sequence's dv infinite, and no other entry of any dv."""
    H, lengths = 2, [5, 33, 16]
    q, k, v, _, _, _, _, meta = _case(device, D, H, lengths, [1, 1, 1], D, grad=True)
    out = flash_attn_mlm_compressed(q, k, v, H, meta, D ** -0.5, block_n=64)
    dout = torch.randn(out.shape, generator=torch.Generator().manual_seed(1)).to(device)
    (want,) = torch.autograd.grad(out, [v], dout, retain_graph=True)
    dout[lengths[0] - 1, 3] = float("inf")  # head 0, sequence 0, its last row
    (got,) = torch.autograd.grad(out, [v], dout)
    want = want.clone()
    want[0, 0, :lengths[0], 3] = float("inf")
    assert torch.equal(got, want)

def _overflowing(device, D, n_keys, hidden, seed):
    """One head of 9 queries over n_keys context keys.  Query 4's score with the first
    `hidden` keys overflows to -inf (key entry 3e38 against -1e10), the others' do not."""
    gen = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn((1, 1, 9, D), generator=gen).to(device) for _ in range(3))
    kc, vc = (torch.randn((n_keys, D), generator=gen).to(device) for _ in range(2))
    q[..., 0] = 0.0
    q[0, 0, 4, 0] = -1e10
    k[..., 0] = 0.0
    kc[:, 0] = 0.0
    kc[:hidden, 0] = 3e38
    return q, k, v, kc, vc


@pytest.mark.parametrize("all_hidden", [False, True])
@pytest.mark.parametrize("D,C", [(32, 40), (64, 100), (64, 5000), (256, 3000)])  # the last two are split
def test_f32_scores_of_minus_infinity(D, C, all_hidden, device):
    """Keys of score -inf have weight 0, also a whole tile or part of them; a row without any
    other key has no softmax: NaN, and the other rows are not touched."""
    q, k, v, kc, vc = _overflowing(device, D, C, C if all_hidden else C - C // 5, D)
    if all_hidden:
        k[..., 0] = 3e38
    cache = InferenceCache()
    cache.prefill_kv_cache(0, k_cache=kc, v_cache=vc, context_batch_size=1, is_mla=False, num_heads=1, head_dim=D)
    out = flash_attn_mlm(q, k, v, D ** -0.5, inference_cache=cache, layer_id=0)
    kk, vv = torch.cat([kc, k[0, 0]]).double(), torch.cat([vc, v[0, 0]]).double()
    z = (q[0, 0].double() @ kk.T * D ** -0.5).float().double()  # -3e48 is -inf in float32
    ref = torch.softmax(z, dim=-1) @ vv
    assert bool(torch.isnan(ref[4]).all()) == all_hidden and not torch.isnan(ref[[0, 8]]).any()
    torch.testing.assert_close(out[0, 0].double(), ref, atol=TOL, rtol=TOL, equal_nan=True)
