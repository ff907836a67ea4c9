"""The work that a user of this package has it do, as cases that can be timed.

Every case goes through a public entry point: ``flash_naylis_attn`` (training:
forward and backward; prefill: forward alone), ``flash_naylis_decode``,
``rope_varlen`` (QK-RMSNorm and RoPE of a pack, forward and backward) and
``NaylisAttention`` (a whole layer: a training step on a pack, and a decode
step against a ``StaticKVCache``).  ``listed()`` holds the named ones,
``draw()`` makes more of the same ranges: 1 to 64 sequences, lengths from 16
to 16384, head dims 64 and 128, ranks 8 to 64, grouped and ungrouped heads,
vanilla heads beside graph heads, bf16 and fp16, causal and not, dense and
packed.  ``exact()`` restates the same operations in 64 bits with plain torch.
"""
import math

import torch

from fna2_amd.attention_fna2 import NaylisAttention, StaticKVCache
from fna2_amd.decode import flash_naylis_decode
from fna2_amd.flash_naylis_attn import flash_naylis_attn
from fna2_amd.rope import rope_varlen

_DT = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def listed():
    return [
        # A layer's attention at a small model's sizes (the reference's
        # large_seq validation shape): one short sequence, grouped heads,
        # half the heads without a bias.  Latency and launches.
        dict(name="train_small", kind="train", pack=False, B=1, H=8, HKV=4, HG=4, D=64, R=32,
             L=512, causal=True, dtype="bf16"),
        # Pre-training of a small model: a batch of ordinary sequences.
        dict(name="train_batch", kind="train", pack=False, B=4, H=16, HKV=16, HG=16, D=64, R=16,
             L=2048, causal=True, dtype="bf16"),
        # Packed pre-training, the headline workload: 64 documents of 64 to
        # 512 tokens, 16384 in all.
        dict(name="train_pack", kind="train", pack=True, B=64, H=16, HKV=16, HG=16, D=128, R=32,
             L=16384, lo=64, hi=512, causal=True, dtype="bf16"),
        # Long-context training.
        dict(name="train_long", kind="train", pack=False, B=1, H=32, HKV=32, HG=32, D=128, R=64,
             L=16384, causal=True, dtype="bf16"),
        # An encoder's pack: one very long document beside many short ones,
        # not causal.
        dict(name="train_skewed", kind="train", pack=True, B=385, H=8, HKV=8, HG=8, D=64, R=16,
             L=32768, lo=16, hi=128, long=8192, causal=False, dtype="bf16"),
        # fp16 training with grouped and vanilla heads at an odd length.
        dict(name="train_gqa_fp16", kind="train", pack=False, B=2, H=16, HKV=4, HG=12, D=128, R=24,
             L=1531, causal=True, dtype="fp16"),
        # Serving, prompt: one odd-length prompt through grouped heads,
        # forward alone.
        dict(name="prefill", kind="prefill", pack=False, B=1, H=32, HKV=8, HG=32, D=128, R=32,
             L=3001, causal=True, dtype="bf16"),
        # Serving, one token for each of 64 sequences, bias from a cached R_k.
        dict(name="decode_batch", kind="decode", B=64, H=16, HKV=16, HG=16, D=128, R=32, L=4096,
             ragged=False, dtype="bf16"),
        # Serving, few ragged sequences, grouped heads, no bias: latency.
        dict(name="decode_few", kind="decode", B=4, H=32, HKV=8, HG=0, D=128, R=0, L=2500,
             ragged=True, dtype="bf16"),
        # QK-RMSNorm and RoPE of the packed workload, forward and backward.
        dict(name="norm_rope_pack", kind="rope", B=64, H=16, HKV=16, D=128, L=16384, lo=64, hi=512,
             dtype="bf16"),
        # One whole layer's training step on the packed workload.
        dict(name="layer_train", kind="layer", pack=True, B=64, E=2048, H=16, HKV=16, R=32,
             L=16384, lo=64, hi=512, dtype="bf16"),
        # One whole layer's decode step against a preallocated cache, with
        # the bias.
        dict(name="layer_decode", kind="layer_decode", B=16, E=2048, H=16, HKV=16, R=32, L=2047,
             dtype="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _heads(rng):
    h, kv = rng.choice([(8, 4), (8, 8), (12, 4), (16, 16), (16, 4), (32, 8), (32, 32)])
    g = rng.choice([h, h, h // 2, 3 * h // 4])
    return dict(H=h, HKV=kv, HG=g)


def draw(rng):
    kind = rng.choice(["train", "train", "train", "prefill", "decode", "decode", "rope", "layer",
                       "layer_decode"])
    if kind in ("train", "prefill"):
        pack = rng.random() < 0.4
        c = dict(kind=kind, pack=pack, **_heads(rng), D=rng.choice([64, 128]),
                 R=rng.choice([8, 16, 24, 32, 32, 64]), causal=rng.random() < 0.75,
                 dtype=rng.choice(["bf16", "bf16", "bf16", "fp16"]))
        if pack:
            lo, hi = sorted((_log(rng, 16, 2048), _log(rng, 64, 4096)))
            n = _log(rng, 2, 64)
            long = rng.choice([0, 0, _log(rng, 1024, 8192)])
            n = max(2, min(n, (32768 - long) // hi))
            mid = sum(divmod(n * (lo + hi), 2))
            return dict(c, B=n + (long > 0), L=mid + long, lo=lo, hi=hi, long=long)
        c["L"] = _log(rng, 64, 8192)
        c["B"] = max(1, min(_log(rng, 1, 16), 32768 // c["L"]))
        while c["B"] > 1 and work(c)["flops"] > 9e12:  # (train_long's: 9.9e12)
            c["B"] -= 1
        return c
    if kind == "decode":
        bias = rng.random() < 0.5
        c = dict(kind=kind, **_heads(rng), D=rng.choice([64, 128]), R=rng.choice([16, 32, 32]),
                 B=_log(rng, 1, 64), L=_log(rng, 64, 8192), ragged=rng.random() < 0.5,
                 dtype="bf16")
        if not bias:
            c.update(HG=0, R=0)
        c["L"] = min(c["L"], 64 * 4096 * 16 // (c["B"] * c["HKV"]))
        return c
    if kind == "rope":
        h = _heads(rng)
        lo = _log(rng, 16, 512)
        hi, n = 2 * lo, _log(rng, 1, 64)
        return dict(kind=kind, B=n, H=h["H"], HKV=h["HKV"], D=rng.choice([64, 128]),
                    L=n * (lo + hi) // 2, lo=lo, hi=hi, dtype=rng.choice(["bf16", "bf16", "fp32"]))
    E, H = rng.choice([(512, 8), (1024, 16), (1024, 8), (2048, 16)])
    c = dict(kind=kind, E=E, H=H, HKV=rng.choice([H, H // 2, H // 4]), R=rng.choice([16, 32]),
             dtype="bf16")
    if kind == "layer":
        lo = _log(rng, 32, 512)
        hi, n = 2 * lo, _log(rng, 2, 64)
        n = min(n, 16384 // hi)
        return dict(c, pack=rng.random() < 0.5, B=n, L=n * (lo + hi) // 2, lo=lo, hi=hi)
    return dict(c, B=_log(rng, 1, 64), L=_log(rng, 33, 4095))


# -- the sizes of a case ------------------------------------------------------

def _lengths(case):
    """The lengths of a pack: the long document (if any) first, the others
    spread over [lo, hi] by a fixed odd stride and nudged to the total."""
    n, total, lo, hi = case["B"], case["L"], case["lo"], case["hi"]
    long = case.get("long", 0)
    head = [long] if long else []
    n -= len(head)
    rest = total - sum(head)
    span = hi - lo + 1
    lens = [lo + (i * 7919 + 13) % span for i in range(n)]
    i, off = 0, rest - sum(lens)
    while off and i < 8 * n:
        new = min(max(lens[i % n] + math.ceil(off / max(n - i % n, 1)), lo), hi)
        off -= new - lens[i % n]
        lens[i % n] = new
        i += 1
    lens[-1] += off  # (a total outside n * [lo, hi])
    return head + lens


def _seqs(case):
    """The lengths of a case's sequences."""
    if case["kind"] == "rope" or case.get("pack"):
        return _lengths(case)
    if case["kind"] == "layer":  # a dense batch of one length
        return [max(case["L"] // case["B"], 1)] * case["B"]
    return [case["L"]] * case["B"]


def _pairs(lens, causal):
    return sum(n * (n + 1) // 2 if causal else n * n for n in lens)


def work(case):
    k = case["kind"]
    es = 4 if case["dtype"] == "fp32" else 2
    H, HKV = case["H"], case["HKV"]
    if k in ("train", "prefill"):
        lens = _seqs(case)
        T, D, R, HG = sum(lens), case["D"], case["R"], case["HG"]
        p = _pairs(lens, case["causal"])
        qkv = T * (H + 2 * HKV) * D * 2 + 2 * T * HG * R * 2
        if k == "prefill":
            return dict(bytes=qkv + T * H * D * 2, flops=p * (H * 4 * D + HG * 2 * R))
        # q, k, v, R read, dO read, out written, and a gradient for each input
        return dict(bytes=2 * qkv + 2 * T * H * D * 2, flops=p * (H * 14 * D + HG * 8 * R))
    if k == "decode":
        rows = sum(_cache_lens(case))
        D, R, HG, B = case["D"], case["R"], case["HG"], case["B"]
        return dict(bytes=rows * (2 * HKV * D + HG * R) * 2 + B * (2 * H * D + HG * R) * 2,
                    flops=rows * (H * 4 * D + HG * 2 * R))
    if k == "rope":
        rows = sum(_seqs(case)) * (H + HKV) * case["D"]
        return dict(bytes=rows * es * 5, flops=rows * 20)
    E, R, D = case["E"], case["R"], case["E"] // H
    width = E + 2 * HKV * D + 2 * H * R
    if k == "layer":
        lens = _seqs(case)
        T = sum(lens)
        mm = 2 * T * E * (width + E)
        return dict(bytes=(4 * T * E + 2 * (width + E) * E) * 2,
                    flops=3 * mm + _pairs(lens, True) * H * (14 * D + 8 * R))
    B, L = case["B"], case["L"]
    return dict(bytes=(E * (width + E) + 2 * B * E) * 2 + B * (L + 1) * (2 * HKV * D + H * R) * 2,
                flops=2 * B * E * (width + E) + B * (L + 1) * H * (4 * D + 2 * R))


def tolerance(case):
    """About four times the error against exact(): one attention call 2.1e-3
    to 2.5e-3 (d_graph_scale, a sum with cancellation, 3.4e-3), the norm and
    rotation 1.7e-3, a layer's step, rounded to bf16 between its parts,
    2.6e-2, and its decode step 6e-3."""
    return {
        "train": {"rel": 0.014, "max": 0.5},
        "prefill": {"rel": 0.01, "max": 0.2},
        "decode": {"rel": 0.01, "max": 0.2},
        "rope": {"rel": 0.007, "max": 0.1},
        "layer": {"rel": 0.03, "max": 0.9},
        "layer_decode": {"rel": 0.02, "max": 0.3},
    }[case["kind"]]


# -- inputs -------------------------------------------------------------------

def _dev():
    return torch.device("cuda", torch.cuda.current_device())


def _gen(seed):
    g = torch.Generator(device=_dev())
    g.manual_seed(seed)
    return g


def _randn(g, *shape, std=1.0, dtype=torch.bfloat16):
    return (torch.randn(*shape, generator=g, device=g.device) * std).to(dtype)


def _cu(lens):
    c = [0]
    for n in lens:
        c.append(c[-1] + n)
    return torch.tensor(c, dtype=torch.int32, device=_dev())


def _cache_lens(case):
    """Rows in use of each sequence's cache (the new token's included)."""
    if not case["ragged"]:
        return [case["L"]] * case["B"]
    lo = max(case["L"] // 3, 1)
    return [case["L"] - (i * 7919) % (case["L"] - lo + 1) for i in range(case["B"])]


def _attn_inputs(case, seed):
    """q, k, v, R_q, R_k, graph_scale, dO: q / k / v / dO as normalised rows
    are, R as the low-rank projections give it (dot products of order one
    for a short rank), packed [T, H, F] or dense [B, H, S, F] views of
    [B, S, H, F] memory, as projections write them."""
    g, dt = _gen(seed), _DT[case["dtype"]]
    H, HKV, HG, D, R = (case[x] for x in ("H", "HKV", "HG", "D", "R"))
    lens = _seqs(case)
    lead = (sum(lens),) if case["pack"] else (case["B"], case["L"])

    def t(h, f, std=1.0, dtype=dt):
        x = _randn(g, *lead, h, f, std=std, dtype=dtype)
        return x if case["pack"] else x.transpose(1, 2)

    rs = R ** -0.5
    return (t(H, D), t(HKV, D), t(HKV, D), t(HG, R, rs, torch.bfloat16),
            t(HG, R, rs, torch.bfloat16), 1.0 + 0.5 * _randn(g, HG, dtype=torch.float32),
            t(H, D), lens)


def _rope_inputs(case, seed):
    g, dt = _gen(seed), _DT[case["dtype"]]
    lens, D = _seqs(case), case["D"]
    T = sum(lens)
    q, k = _randn(g, T, case["H"], D, dtype=dt), _randn(g, T, case["HKV"], D, dtype=dt)
    wq = 1.0 + 0.2 * _randn(g, D, dtype=torch.float32)
    wk = 1.0 + 0.2 * _randn(g, D, dtype=torch.float32)
    gq, gk = _randn(g, T, case["H"], D, dtype=dt), _randn(g, T, case["HKV"], D, dtype=dt)
    inv = _inv_freq(D).to(_dev())
    return q, k, wq, wk, gq, gk, inv, lens


def _inv_freq(D):
    return 1.0 / (10000 ** (torch.arange(0, D, 2, dtype=torch.float32) / D))


def _layer(case, g):
    E, H, HKV, R = (case[x] for x in ("E", "H", "HKV", "R"))
    with torch.device(_dev()):
        m = NaylisAttention(E, H, n_kv_heads=HKV, rel_rank=R, max_seq_len=4096,
                            decode_graph_bias=case["kind"] == "layer_decode")
    m = m.to(torch.bfloat16)
    with torch.no_grad():
        for name, p in m.named_parameters():
            if p.dim() == 2:  # (R's projections: bias terms of order one)
                p.copy_(_randn(g, *p.shape, std=E ** -0.5 * (R ** -0.25 if "rel_" in name else 1)))
            elif name == "graph_scale":
                p.copy_(1.0 + 0.5 * _randn(g, *p.shape))
            else:
                p.copy_(1.0 + 0.2 * _randn(g, *p.shape))
    return m


def prepare(case, seed):
    k = case["kind"]
    if k in ("train", "prefill"):
        q, kk, v, rq, rk, gs, dout, lens = _attn_inputs(case, seed)
        kw = dict(softmax_scale=case["D"] ** -0.5, is_causal=case["causal"])
        if case["pack"]:
            cu = _cu(lens)
            kw.update(cu_seqlens_q=cu, cu_seqlens_k=cu, max_seqlen_q=max(lens),
                      max_seqlen_k=max(lens))
        ins = (q, kk, v, rq, rk, gs)
        if k == "train":
            ins = tuple(t.requires_grad_(True) for t in ins)
        return dict(kind=k, ins=ins, dout=dout, kw=kw)
    if k == "decode":
        g = _gen(seed)
        B, H, HKV, HG, D, R, L = (case[x] for x in ("B", "H", "HKV", "HG", "D", "R", "L"))
        kw = dict(softmax_scale=D ** -0.5)
        if case["ragged"]:
            kw["cache_seqlens"] = torch.tensor(_cache_lens(case), dtype=torch.int32, device=_dev())
        ins = [_randn(g, B, H, D), _randn(g, B, HKV, L, D), _randn(g, B, HKV, L, D)]
        if HG:
            ins += [_randn(g, B, HG, R, std=R ** -0.5), _randn(g, B, HG, L, R, std=R ** -0.5),
                    1.0 + 0.5 * _randn(g, HG, dtype=torch.float32)]
        return dict(kind=k, ins=ins, kw=kw)
    if k == "rope":
        q, kk, wq, wk, gq, gk, inv, lens = _rope_inputs(case, seed)
        ins = tuple(t.requires_grad_(True) for t in (q, kk, wq, wk))
        return dict(kind=k, ins=ins, cu=_cu(lens), inv=inv, gout=(gq, gk))
    g = _gen(seed)
    m = _layer(case, g)
    E = case["E"]
    if k == "layer":
        lens = _seqs(case)
        T = sum(lens)
        kw = {}
        shape = (case["B"], lens[0], E)
        if case["pack"]:
            cu = _cu(lens)
            shape = (T, E)
            kw = dict(cu_seqlens_q=cu, cu_seqlens_k=cu, max_seqlen_q=max(lens),
                      max_seqlen_k=max(lens))
        x = _randn(g, *shape).requires_grad_(True)
        return dict(kind=k, m=m, x=x, dy=_randn(g, *shape), kw=kw,
                    params=[p for p in m.parameters()])
    m = m.eval()
    B, L, H, HKV, R, D = case["B"], case["L"], case["H"], case["HKV"], case["R"], E // case["H"]
    cache = StaticKVCache.empty(B, HKV, L + 1, D, H, R, device=_dev())
    cache.append(*_cached_rows(case, g))
    return dict(kind=k, m=m, x=_randn(g, B, 1, E), cache=cache, L=L)


def _cached_rows(case, g):
    B, L, H, HKV, R = case["B"], case["L"], case["H"], case["HKV"], case["R"]
    D = case["E"] // H
    return (_randn(g, B, HKV, L, D), _randn(g, B, HKV, L, D),
            _randn(g, B, H, L, R, std=R ** -0.25))


# -- one pass -----------------------------------------------------------------

def run(state):
    k = state["kind"]
    if k == "train":
        out = flash_naylis_attn(*state["ins"], **state["kw"])
        return (out, *torch.autograd.grad(out, state["ins"], state["dout"]))
    if k == "prefill":
        with torch.no_grad():
            return flash_naylis_attn(*state["ins"], **state["kw"])
    if k == "decode":
        return flash_naylis_decode(*state["ins"], **state["kw"], return_lse=True)
    if k == "rope":
        q, kk, wq, wk = state["ins"]
        outs = rope_varlen(q, kk, state["cu"], state["inv"], wq, wk)
        return (*outs, *torch.autograd.grad(outs, state["ins"], state["gout"]))
    if k == "layer":
        y, _ = state["m"](state["x"], **state["kw"])
        return (y, *torch.autograd.grad(y, [state["x"], *state["params"]], state["dy"]))
    # layer_decode: the same step again on a repeated pass
    cache, n = state["cache"], state["L"]
    cache.length = n
    with torch.no_grad():
        y, _ = state["m"](state["x"], past_kv=cache, use_kv_cache=True)
    # the output, and the rows the step appended
    return y, cache.k[:, :, n:], cache.v[:, :, n:], cache.r_k[:, :, n:]


# -- the same in 64 bits ------------------------------------------------------

_BIG = 1 << 28  # scores of one block


def _attn64(q, k, v, rq, rk, gs, scale, causal, dout=None):
    """Attention of one sequence, [H, S, F] tensors in 64 bits; with dout
    also the gradients.  Heads go in blocks that bound the scores' memory."""
    H, S, D = q.shape
    HKV, HG = k.shape[0], rq.shape[0]
    grp = H // HKV
    out = torch.empty_like(q)
    if dout is not None:
        dq, dk, dv = torch.zeros_like(q), torch.zeros_like(k), torch.zeros_like(v)
        drq, drk, dgs = torch.zeros_like(rq), torch.zeros_like(rk), torch.zeros_like(gs)
    mask = None
    if causal:
        i = torch.arange(S, device=q.device)
        mask = i[None, :] > i[:, None]
    step = max(1, min(H, _BIG // max(S * S, 1)))
    for a in range(0, H, step):
        b = min(a + step, H)
        g = min(max(HG - a, 0), b - a)  # graph heads of the block: its first g
        kv = torch.arange(a, b, device=q.device) // grp
        kb, vb = k[kv], v[kv]
        s = scale * torch.bmm(q[a:b], kb.transpose(1, 2).contiguous())
        if g:
            bias = torch.bmm(rq[a:a + g], rk[a:a + g].transpose(1, 2).contiguous())
            s[:g] += gs[a:a + g, None, None] * bias
        if mask is not None:
            s.masked_fill_(mask, -math.inf)
        p = torch.softmax(s, dim=-1)
        del s
        out[a:b] = torch.bmm(p, vb)
        if dout is None:
            continue
        do = dout[a:b]
        ds = torch.bmm(do, vb.transpose(1, 2).contiguous())
        ds -= (do * out[a:b]).sum(-1, keepdim=True)
        ds *= p
        dv.index_add_(0, kv, torch.bmm(p.transpose(1, 2).contiguous(), do))
        del p
        dst = ds.transpose(1, 2).contiguous()
        dq[a:b] = scale * torch.bmm(ds, kb)
        dk.index_add_(0, kv, scale * torch.bmm(dst, q[a:b]))
        if g:
            w = gs[a:a + g, None, None]
            drq[a:a + g] = w * torch.bmm(ds[:g], rk[a:a + g])
            drk[a:a + g] = w * torch.bmm(dst[:g], rq[a:a + g])
            dgs[a:a + g] = (ds[:g] * bias).sum((1, 2))
    return (out,) if dout is None else (out, dq, dk, dv, drq, drk, dgs)


def _attn64_all(ins, gs, lens, scale, causal, dout=None):
    """_attn64 over a pack: [T, H, F] tensors; the results are packed again."""
    d = torch.float64
    outs = None
    t0 = 0
    dgs = torch.zeros_like(gs, dtype=d)
    for n in lens:
        part = [t[t0:t0 + n].to(d).transpose(0, 1).contiguous() for t in ins]
        do = None if dout is None else dout[t0:t0 + n].to(d).transpose(0, 1).contiguous()
        r = _attn64(*part, gs.to(d), scale, causal, do)
        if outs is None:
            shapes = [ins[0]] if dout is None else [ins[0], *ins]
            outs = [torch.empty(t.shape, dtype=d, device=t.device) for t in shapes]
        for o, x in zip(outs, r):
            o[t0:t0 + n] = x.transpose(0, 1)
        if dout is not None:
            dgs += r[-1]
        t0 += n
    return (*outs, dgs) if dout is not None else tuple(outs)


class _Attn64(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, v, rq, rk, gs, lens, scale):
        ctx.save_for_backward(q, k, v, rq, rk, gs)
        ctx.rest = lens, scale
        return _attn64_all((q, k, v, rq, rk), gs, lens, scale, True)[0]

    @staticmethod
    def backward(ctx, dout):
        q, k, v, rq, rk, gs = ctx.saved_tensors
        r = _attn64_all((q, k, v, rq, rk), gs, *ctx.rest, True, dout)
        return (*r[1:], None, None)


def _rope64(x, ang):
    """Rotates rows [T, H, D] by the angles [T, D / 2]."""
    h = x.shape[-1] // 2
    c, s = ang.cos()[:, None], ang.sin()[:, None]
    a, b = x[..., :h], x[..., h:]
    return torch.cat((a * c - b * s, b * c + a * s), -1)


def _norm64(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * w


def _norm_rope64(q, k, wq, wk, lens, inv):
    pos = torch.cat([torch.arange(n, device=q.device) for n in lens]).to(torch.float64)
    ang = pos[:, None] * inv.to(torch.float64)
    return _rope64(_norm64(q, wq), ang), _rope64(_norm64(k, wk), ang)


def exact(case, seed):
    k = case["kind"]
    d = torch.float64
    if k in ("train", "prefill"):
        *ins, gs, dout, lens = _attn_inputs(case, seed)
        back = k == "train"
        if not case["pack"]:  # one sequence after the other
            ins = [t.transpose(1, 2).flatten(0, 1) for t in ins]
            dout = dout.transpose(1, 2).flatten(0, 1)
        r = _attn64_all(ins, gs, lens, case["D"] ** -0.5, case["causal"], dout if back else None)
        if not case["pack"]:
            r = [t if t.dim() == 1 else t.view(case["B"], case["L"], *t.shape[1:]).transpose(1, 2)
                 for t in r]
        return tuple(r) if back else r[0]
    if k == "decode":
        s = prepare(case, seed)
        q, kc, vc = (t.to(d) for t in s["ins"][:3])
        grp = case["H"] // case["HKV"]
        outs, lses = [], []
        for b, n in enumerate(_cache_lens(case)):
            kb = kc[b, :, :n].repeat_interleave(grp, 0)
            vb = vc[b, :, :n].repeat_interleave(grp, 0)
            sc = s["kw"]["softmax_scale"] * (kb * q[b][:, None]).sum(-1)
            if case["HG"]:
                rq, rk, gs = (t.to(d) for t in (s["ins"][3][b], s["ins"][4][b, :, :n], s["ins"][5]))
                sc[:case["HG"]] += gs[:, None] * (rk * rq[:, None]).sum(-1)
            lses.append(torch.logsumexp(sc, -1))
            outs.append((torch.softmax(sc, -1)[..., None] * vb).sum(1))
        return torch.stack(outs), torch.stack(lses)
    if k == "rope":
        q, kk, wq, wk, gq, gk, inv, lens = _rope_inputs(case, seed)
        ins = [t.to(d).requires_grad_(True) for t in (q, kk, wq, wk)]
        with torch.enable_grad():
            outs = _norm_rope64(*ins, lens, inv)
            gr = torch.autograd.grad(outs, ins, (gq.to(d), gk.to(d)))
        return tuple(t.detach() for t in outs) + tuple(gr)
    E, H, HKV, R = (case[x] for x in ("E", "H", "HKV", "R"))
    D = E // H
    s = prepare(case, seed)
    w = {n: p.detach().to(d).requires_grad_(True) for n, p in s["m"].named_parameters()}
    x = s["x"].detach().to(d).requires_grad_(True)

    def project():
        f = x.reshape(-1, E)
        y = [f @ w[n + ".weight"].t() for n in ("q_proj", "k_proj", "v_proj", "rel_q_proj",
                                                "rel_k_proj")]
        return [t.view(f.shape[0], -1, n) for t, n in zip(y, (D, D, D, R, R))]

    inv = _inv_freq(D).to(x.device)
    if k == "layer":
        lens = _seqs(case)
        with torch.enable_grad():
            q, kk, v, rq, rk = project()
            q, kk = _norm_rope64(q, kk, w["q_norm.weight"], w["k_norm.weight"], lens, inv)
            o = _Attn64.apply(q, kk, v, rq, rk, w["graph_scale"], lens, D ** -0.5)
            y = (o.reshape(-1, E) @ w["out_proj.weight"].t()).view(x.shape)
            gr = torch.autograd.grad(y, [x, *w.values()], s["dy"].to(d))
        return (y.detach(), *gr)
    # (the rotary table of a decode step is the module's own: angles formed
    # and kept in the activations' type)
    B, L = case["B"], case["L"]
    with torch.no_grad():
        q, kk, v, rq, rk = project()
        low = torch.bfloat16
        ang = (torch.tensor([L], device=x.device, dtype=low) * inv.to(low))[None]
        cs, sn = ang.cos().to(d)[:, None], ang.sin().to(d)[:, None]

        def rot(t):
            a, b = t[..., :D // 2], t[..., D // 2:]
            return torch.cat((a * cs - b * sn, b * cs + a * sn), -1)

        q = rot(_norm64(q, w["q_norm.weight"]))
        kk = rot(_norm64(kk, w["k_norm.weight"]))
        ck, cv, cr = (t[:, :, :L] for t in (s["cache"].k, s["cache"].v, s["cache"].r_k))
        outs = []
        for b in range(B):
            kb = torch.cat((ck[b].to(d), kk[b][:, None]), 1).repeat_interleave(H // HKV, 0)
            vb = torch.cat((cv[b].to(d), v[b][:, None]), 1).repeat_interleave(H // HKV, 0)
            rb = torch.cat((cr[b].to(d), rk[b][:, None]), 1)
            sc = D ** -0.5 * (kb * q[b][:, None]).sum(-1)
            sc += w["graph_scale"][:, None] * (rb * rq[b][:, None]).sum(-1)
            outs.append((torch.softmax(sc, -1)[..., None] * vb).sum(1))
        y = (torch.stack(outs).view(B, E) @ w["out_proj.weight"].t()).view(B, 1, E)
    return y, kk[:, :, None], v[:, :, None], rk[:, :, None]
