"""The work that users of this framework have it do, as cases that can be timed and checked.

A case is one pass through the public entry points, with everything that a program keeps
between calls (inputs, pack metadata, cached contexts) prepared before it.  ``listed()``
holds one case for each way the framework is used; ``draw()`` gives more of the same ways
at other sizes.  ``exact()`` restates a case in plain torch at 64 bits.

Ways (``case["way"]``):
  dense        flash_attn_mlm over [B, H, N, D], optionally with a shared cached context
  packed       flash_attn_mlm_compressed over ragged sequences, then unpack_from_kernel
  mla          the same with one latent head serving as K and V of all query heads
  ingest       build_pack_metadata, a prefill call that stores its K/V as a layer's
               context, then append_kv_cache of a second chunk
  train        flash_attn_mlm_compressed and its gradients
"""

from __future__ import annotations

import math
import random
import sys
from pathlib import Path

import torch

_PKG = str(Path(__file__).resolve().parent.parent / "flash-mlm_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import flash_mlm as fm  # noqa: E402

_DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
_PAGE = 64


def _case(way, dtype, B, H, N, D, *, lo=0, ctx="none", ctx_lo=0, ctx_hi=0, causal=False, paged=False, lens=0, name=None):
    """lo: shortest sequence (the longest is N; unused for dense); ctx: "none", "shared"
    (one context for all sequences) or "each", of ctx_lo to ctx_hi rows; lens: seed of the
    lengths."""
    c = dict(way=way, dtype=dtype, B=B, H=H, N=N, D=D, lo=lo, ctx=ctx, ctx_lo=ctx_lo, ctx_hi=ctx_hi, causal=causal,
             paged=paged, lens=lens)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest call: a single-precision check of a model's attention, where latency counts
        _case("dense", "fp32", 2, 8, 128, 64, name="dense_fp32_small"),
        # an encoder layer whose batch attends to one prefilled prompt beside its own tokens
        _case("dense", "bf16", 8, 16, 512, 64, ctx="shared", ctx_lo=2048, ctx_hi=2048, name="dense_bf16_prompt"),
        # a few masked positions refined against a long shared document (latency of one user)
        _case("dense", "bf16", 1, 16, 24, 128, ctx="shared", ctx_lo=6000, ctx_hi=6000, name="dense_bf16_infill"),
        # the headline: ragged batch, every sequence with a cached context of its own
        _case("packed", "fp16", 32, 16, 1024, 128, lo=256, ctx="each", ctx_lo=512, ctx_hi=2048, lens=3,
              name="packed_fp16_ctx"),
        # block-causal decoding of a document in segments over a shared context
        _case("packed", "bf16", 16, 12, 512, 64, lo=64, ctx="shared", ctx_lo=4096, ctx_hi=4096, causal=True, lens=4,
              name="packed_bf16_causal"),
        # serving: many users, a few new tokens each, long contexts in a paged pool
        _case("packed", "bf16", 24, 16, 16, 128, lo=1, ctx="each", ctx_lo=500, ctx_hi=6000, paged=True, lens=5,
              name="packed_bf16_serving"),
        # MLA encoder pass: 64 query heads over one 512-wide latent, cached latents (the largest)
        _case("mla", "bf16", 4, 64, 2048, 512, lo=512, ctx="each", ctx_lo=8192, ctx_hi=8192, lens=6,
              name="mla_bf16_encode"),
        # MLA serving: one to four new tokens a sequence against long cached latents
        _case("mla", "bf16", 16, 64, 4, 512, lo=1, ctx="each", ctx_lo=1000, ctx_hi=8192, lens=7,
              name="mla_bf16_serving"),
        # a document batch is taken in: metadata, prefill into the cache, a second chunk appended
        _case("ingest", "fp16", 16, 16, 1024, 128, lo=256, lens=8, name="ingest_fp16"),
        # a training step's attention: ragged fp16 batch, gradients of q, k, v and the context
        _case("train", "fp16", 32, 16, 1024, 128, lo=256, ctx="each", ctx_lo=512, ctx_hi=2048, lens=3,
              name="train_fp16_ctx"),
        # masked-language-model training, ragged batch without a context
        _case("train", "bf16", 32, 12, 512, 64, lo=64, lens=10, name="train_bf16_mlm"),
        # single-precision training
        _case("train", "fp32", 8, 12, 512, 64, lo=64, lens=11, name="train_fp32"),
    ]


def draw(rng: random.Random):
    def size(lo, hi):  # spread over the logarithm
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    way = rng.choice(["dense", "dense", "packed", "packed", "packed", "mla", "ingest", "train", "train", "train"])
    lens = rng.randrange(1 << 30)
    if way == "mla":
        if rng.random() < 0.5:  # serving
            N = rng.randint(1, 8)
            lo = rng.randint(500, 8000)
            return _case(way, rng.choice(["bf16", "fp16"]), size(1, 48), rng.choice([16, 32, 64]), N, 512,
                         lo=rng.randint(1, N), ctx="each", ctx_lo=lo, ctx_hi=rng.randint(lo, 8192),
                         paged=rng.random() < 0.3, lens=lens)
        N = size(64, 2048)
        lo = rng.randint(256, 4096)
        return _case(way, rng.choice(["bf16", "fp16"]), rng.randint(1, 4), rng.choice([16, 32, 64]), N, 512,
                     lo=rng.randint(1, N), ctx="each", ctx_lo=lo, ctx_hi=rng.randint(lo, 8192), lens=lens)
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp16", "fp32"])
    D = rng.choice([32, 64, 64, 128, 128, 256])
    H = rng.choice([4, 8, 12, 16])
    most = 8 if D == 256 or dtype == "fp32" else 32  # sequences
    ctx = "none" if way == "ingest" else rng.choice(["none", "shared", "each"])
    if way == "dense":
        if ctx == "each":
            ctx = "shared"
        N, B, C = size(8, 1024), min(most, size(1, 16)), size(64, 8192)
        if dtype == "fp32":
            N, C = min(N, 600), min(C, 2048)
        return _case(way, dtype, B, H, N, D, ctx=ctx, ctx_lo=C, ctx_hi=C)
    serving = way == "packed" and rng.random() < 0.4
    N = size(1, 64) if serving else size(32, 1024)
    B = size(1, 64) if serving else min(most, size(1, 32))
    lo = rng.randint(1, N)
    c0 = size(64, 4096)
    c1 = rng.randint(c0, 2 * c0)
    if dtype == "fp32":
        N, B, c0, c1 = min(N, 600), min(B, 8), min(c0, 1024), min(c1, 1024)
        lo = min(lo, N)
    if ctx == "shared":
        c1 = c0
    causal = way == "packed" and ctx != "each" and rng.random() < 0.4
    paged = way == "packed" and ctx == "each" and dtype != "fp32" and rng.random() < 0.4
    return _case(way, dtype, B, H, N, D, lo=lo, ctx=ctx, ctx_lo=c0 if ctx != "none" else 0,
                 ctx_hi=c1 if ctx != "none" else 0, causal=causal, paged=paged, lens=lens)


# ---------------------------------------------------------------------------
# sizes and inputs
# ---------------------------------------------------------------------------
def _dense(case):
    return case["way"] == "dense"


def _train(case):
    return case["way"] == "train"


def _lengths(case):
    """(query lengths, context lengths: one per context batch, [] without a context)"""
    r = random.Random(case["lens"])
    B, N = case["B"], case["N"]
    lq = [N] * B if _dense(case) else [r.randint(case["lo"], N) for _ in range(B)]
    if case["ctx"] == "none":
        return lq, []
    n = 1 if case["ctx"] == "shared" else B
    return lq, [r.randint(case["ctx_lo"], case["ctx_hi"]) for _ in range(n)]


def _pairs(case):
    """Query-key pairs of one head."""
    lq, lc = _lengths(case)
    total, seen = 0, 0
    for b, n in enumerate(lq):
        seen += n
        ctx = (lc[b] if len(lc) > 1 else lc[0]) if lc else 0
        total += n * (ctx + (seen if case["causal"] else n))
    return total


def _randn(gen, shape, dtype, std):
    return (torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32) * std).to(dtype)


def _inputs(case, seed):
    """q, k, v, context rows (head-major), and for training the output's gradient; for
    ingest the chunk that is appended."""
    dt, (B, H, N, D) = _DTYPES[case["dtype"]], (case["B"], case["H"], case["N"], case["D"])
    mla = case["way"] == "mla"
    std = 0.5 if mla else 1.0
    lq, lc = _lengths(case)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    hk = 1 if mla else H
    x = {"q": _randn(gen, (B, H, N, D), dt, std)}
    if mla:  # one latent head, shaped like q without copies
        x["k"] = x["v"] = _randn(gen, (B, 1, N, D), dt, std).expand(B, H, N, D)
    else:
        x["k"], x["v"] = _randn(gen, (B, H, N, D), dt, std), _randn(gen, (B, H, N, D), dt, std)
    if lc:
        x["kc"] = _randn(gen, (hk * sum(lc), D), dt, std)
        x["vc"] = None if mla else _randn(gen, (hk * sum(lc), D), dt, std)
    if case["way"] == "ingest":  # the second chunk: 32 rows a sequence
        x["ka"], x["va"] = _randn(gen, (H * B * 32, D), dt, std), _randn(gen, (H * B * 32, D), dt, std)
    if _train(case):
        x["dout"] = _randn(gen, (H * sum(lq), D), dt, std)
    return x


def _prefix(xs):
    out = [0]
    for n in xs:
        out.append(out[-1] + n)
    return out


def _i32(xs):
    return torch.tensor(xs, dtype=torch.int32, device="cuda")


def _store_pages(cache, x, lc, H, D, mla, lens):
    """The context rows in a pool of 64-row pages, in an order of their own."""
    hk = 1 if mla else H
    need = [(n + _PAGE - 1) // _PAGE for n in lc]
    order = list(range(sum(need)))
    random.Random(lens + 1).shuffle(order)
    table = torch.zeros((len(lc), max(need)), dtype=torch.int32)
    src, dst, first = [], [], 0
    cu = _prefix(lc)
    for c, (n, pages) in enumerate(zip(lc, need)):
        table[c, :pages] = torch.tensor(order[first:first + pages], dtype=torch.int32)
        first += pages
        j = torch.arange(n)
        src.append(cu[c] + j)
        dst.append(table[c].long()[j // _PAGE] * _PAGE + j % _PAGE)
    src, dst = torch.cat(src).cuda(), torch.cat(dst).cuda()

    def pool(rows):
        p = torch.zeros((hk, sum(need) * _PAGE, D), dtype=rows.dtype, device="cuda")
        p[:, dst] = rows.view(hk, -1, D)[:, src]
        return p.view(hk, sum(need), _PAGE, D)

    cache.prefill_paged_kv_cache(0, k_pages=pool(x["kc"]), v_pages=None if mla else pool(x["vc"]),
                                 block_table=table.cuda(), context_lens=torch.tensor(lc, dtype=torch.int32),
                                 is_mla=mla, num_heads=H, head_dim=D)


def prepare(case, seed):
    H, N, D = case["H"], case["N"], case["D"]
    mla = case["way"] == "mla"
    lq, lc = _lengths(case)
    x = _inputs(case, seed)
    s = {"case": case, "x": x, "scale": 1.0 / math.sqrt(D), "cache": fm.InferenceCache(), "lengths": _i32(lq)}
    if _train(case):
        s["leaves"] = [x[n].requires_grad_() for n in ("q", "k", "v", "kc", "vc") if n in x]
    if lc and case["paged"]:
        _store_pages(s["cache"], x, lc, H, D, mla, case["lens"])
    elif lc and _dense(case):
        s["cache"].prefill_kv_cache(0, k_cache=x["kc"], v_cache=x["vc"], context_batch_size=1, is_mla=mla,
                                    num_heads=H, head_dim=D)
    elif lc:
        s["cache"].prefill_kv_cache(0, k_cache=x["kc"], v_cache=x["vc"], total_context_len=sum(lc),
                                    cu_seqlens_kv=_i32(_prefix(lc)), context_batch_size=len(lc), is_mla=mla,
                                    num_heads=H, head_dim=D)
    if not _dense(case) and case["way"] != "ingest":
        s["meta"] = s["cache"].packing.get_pack_metadata(s["lengths"], N=N, block_n=64)
    if case["way"] == "ingest":
        s["cu_add"] = _i32(_prefix([32] * case["B"]))
    return s


def run(s):
    case, x, H = s["case"], s["x"], s["case"]["H"]
    way = case["way"]
    if way == "dense":
        out = fm.flash_attn_mlm(x["q"], x["k"], x["v"], s["scale"], inference_cache=s["cache"], layer_id=0)
    elif way == "ingest":
        meta = fm.build_pack_metadata(s["lengths"], case["N"], 64)
        out = fm.flash_attn_mlm_compressed(x["q"], x["k"], x["v"], H, meta, s["scale"], s["cache"], 0, block_n=64,
                                           prefill=True)
        s["cache"].append_kv_cache(0, k_cache=x["ka"], v_cache=x["va"], cu_seqlens_kv=s["cu_add"])
        e = s["cache"].layer_entry(0)
        return {"out": out, "k_cache": e.k_cache, "v_cache": e.v_cache, "cu_seqlens_kv": e.cu_seqlens_kv}
    else:
        out = fm.flash_attn_mlm_compressed(x["q"], x["k"], x["v"], H, s["meta"], s["scale"], s["cache"], 0,
                                           is_mla=way == "mla", block_n=64, causal_query_seq_attn=case["causal"])
    if _train(case):
        return [out.detach(), *torch.autograd.grad(out, s["leaves"], x["dout"])]
    return out if way == "dense" else fm.unpack_from_kernel(out, s["meta"], H)


def work(case):
    es = torch.finfo(_DTYPES[case["dtype"]]).bits // 8
    B, H, N, D = case["B"], case["H"], case["N"], case["D"]
    mla = case["way"] == "mla"
    lq, lc = _lengths(case)
    T, m = sum(lq), 1 if mla else 2 * H
    elems = 2 * H * T + m * (T + sum(lc))  # q, out, keys and values
    if case["way"] in ("packed", "mla"):
        elems += H * (T + B * N)  # the packed output read again, the padded one written
    elif case["way"] == "ingest":  # the stored rows written, read and written with the chunk's
        elems += 2 * H * (3 * T + 2 * 32 * B)
    flops = 4.0 * H * D * _pairs(case)
    if _train(case):  # dout read with q, k, v, o again; every gradient written
        flops *= 3.5
        elems += 3 * H * T + m * (T + sum(lc)) + H * B * N + m * (B * N + sum(lc))
    return {"bytes": float(es * elems * D), "flops": flops}


def tolerance(case):
    # four times the error against exact() of outputs and gradients over these ranges: up to
    # 8e-7 to 1.2e-6 in fp32, 2.2e-3 to 3.0e-3 in bf16, 3.6e-4 in fp16
    if case["dtype"] == "fp32":
        return {"rel": 5e-6}
    if case["dtype"] == "bf16":
        return {"rel": 1e-2}
    return {"rel": 1.5e-3}


# ---------------------------------------------------------------------------
# the same in plain torch at 64 bits
# ---------------------------------------------------------------------------
def _attend(q, k, v, scale, dout=None):
    """softmax(scale q k^T) v for [h, n, d] queries and [h, m, d] keys, and with dout the
    gradients of q, k and v."""
    p = torch.matmul(q, k.transpose(1, 2).contiguous()).mul_(scale)
    p = torch.softmax(p, dim=-1)
    o = torch.matmul(p, v)
    if dout is None:
        return (o,)
    dv = torch.matmul(p.transpose(1, 2).contiguous(), dout)
    ds = torch.matmul(dout, v.transpose(1, 2).contiguous())
    ds -= (dout * o).sum(-1, keepdim=True)
    ds *= p
    ds *= scale
    return o, torch.matmul(ds, k), torch.matmul(ds.transpose(1, 2).contiguous(), q), dv


def exact(case, seed):
    x = {n: None if t is None else t.double() for n, t in _inputs(case, seed).items() if n not in ("k", "v")}
    raw = _inputs(case, seed)
    B, H, N, D = case["B"], case["H"], case["N"], case["D"]
    mla, dense, train = case["way"] == "mla", _dense(case), _train(case)
    k, v = (raw[n][:, :1 if mla else H].double() for n in ("k", "v"))
    hk = 1 if mla else H
    lq, lc = _lengths(case)
    cu, cuc = _prefix(lq), _prefix(lc)
    T, Tc, scale = cu[-1], cuc[-1], 1.0 / math.sqrt(D)
    kc, vc = (x["kc"].view(hk, Tc, D), (x["kc"] if mla else x["vc"]).view(hk, Tc, D)) if lc else (None, None)
    out = torch.zeros((B, H, N, D), dtype=torch.float64, device="cuda")
    if train:
        g = [torch.zeros_like(out), torch.zeros_like(k), torch.zeros_like(v)]
        gc = [torch.zeros_like(kc), torch.zeros_like(vc)] if lc else []
    for b, n in enumerate(lq):
        c = slice(*(cuc[:2] if len(lc) == 1 else cuc[b:b + 2])) if lc else slice(0, 0)
        first = 0 if case["causal"] else b
        ks = ([kc[:, c]] if lc else []) + [k[i, :, :lq[i]] for i in range(first, b + 1)]
        vs = ([vc[:, c]] if lc else []) + [v[i, :, :lq[i]] for i in range(first, b + 1)]
        kk, vv = torch.cat(ks, 1), torch.cat(vs, 1)
        nc = c.stop - c.start
        step = max(1, int(2e9 // (8 * max(1, n) * kk.shape[1])))  # heads at a time
        for h0 in range(0, H, step):
            hs = slice(h0, min(H, h0 + step))
            kh, vh = (kk.expand(hs.stop - h0, -1, -1), vv.expand(hs.stop - h0, -1, -1)) if mla else (kk[hs], vv[hs])
            d = None
            if train:
                d = x["dout"].view(H, T, D)[hs, cu[b]:cu[b + 1]].contiguous()
            r = _attend(x["q"][b, hs, :n].contiguous(), kh.contiguous(), vh.contiguous(), scale, d)
            out[b, hs, :n] = r[0]
            if train:
                g[0][b, hs, :n] = r[1]
                for gi, gci, ri in zip(g[1:], gc or [None, None], r[2:]):
                    gi[b, hs, :n] += ri[:, nc:]
                    if lc:
                        gci[hs, c] += ri[:, :nc]
    packed = out if dense else torch.cat([out[b, :, :n] for b, n in enumerate(lq)], 1).reshape(H * T, D)
    if train:
        return [packed, *g, *(t.view(hk * Tc, D) for t in gc)]
    if case["way"] == "ingest":
        return {"out": packed, "k_cache": None, "v_cache": None, "cu_seqlens_kv": None}
    return out
