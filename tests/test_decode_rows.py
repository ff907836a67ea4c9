"""fna2_decode_rows: the new token's rows of a decode step (QK-RMSNorm,
rotation, cache append) in one launch, against the formula in fp64, and the
module's step with it against the step by torch modules."""
import ctypes

import pytest
import torch

from fna2_amd import _capi

FAKE = 1 << 20


def _args(**over):
    a = _capi.DecodeRowsArgs()
    a.batch, a.heads, a.heads_kv, a.heads_graph, a.head_dim, a.rank = 2, 8, 4, 6, 128, 24
    for n in ("q", "k", "v", "r_k", "q_out", "k_out", "v_out", "rk_out"):
        setattr(a, n, _capi.Tensor(FAKE, 4096, 0, 128))
    a.norm_q = a.norm_k = a.cos = a.sin = FAKE
    a.eps_q = a.eps_k = 1e-6
    for n, v in over.items():
        setattr(a, n, v)
    return a


@pytest.mark.parametrize("over,status", [
    (dict(), "FNA2_OK"),
    (dict(head_dim=96), "FNA2_E_HEAD_DIM"),
    (dict(heads=0), "FNA2_E_HEADS"),
    (dict(rank=12), "FNA2_E_RANK"),
    (dict(batch=-1), "FNA2_E_SHAPE"),
    (dict(batch=1 << 24), "FNA2_E_SHAPE"),
    (dict(eps_k=float("nan")), "FNA2_E_SCALE"),
    (dict(sin=None), "FNA2_E_NULL"),
    (dict(norm_q=FAKE + 2), "FNA2_E_STRIDE"),
    (dict(k_out=_capi.Tensor(FAKE + 8, 4096, 0, 128)), "FNA2_E_STRIDE"),
    (dict(v=_capi.Tensor(FAKE, 4096, 0, 129)), "FNA2_E_STRIDE"),
    (dict(rk_out=_capi.Tensor(None, 0, 0, 0)), "FNA2_E_NULL"),
    (dict(rk_out=_capi.Tensor(None, 0, 0, 0), heads_graph=0), "FNA2_OK"),
])
def test_check(over, status):
    a = _args(**over)
    assert _capi.STATUS[_capi.lib().fna2_check_decode_rows(ctypes.byref(a))] == status


CASES = [  # B, H, HKV, HG, D, R, norm, rope
    (1, 1, 1, 0, 64, 0, True, True),
    (3, 8, 2, 6, 64, 64, True, True),
    (2, 6, 6, 5, 128, 24, True, False),
    (5, 4, 1, 4, 128, 8, False, True),
    (33, 16, 16, 16, 128, 32, True, True),
    (2, 4, 2, 0, 64, 0, False, False),
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_rows_against_the_formula(gpu, case):
    B, H, HKV, HG, D, R, norm, rope = case
    print(case, flush=True)
    g = torch.Generator().manual_seed(sum(map(int, case)))
    mk = lambda *s: torch.randn(*s, generator=g).bfloat16().to(gpu)
    # one projection output, read as column views; a cache of 7 rows, row 4 written
    wide = mk(B, (H + 2 * HKV) * D + HG * R + 8)
    cut = [0, H * D, (H + HKV) * D, (H + 2 * HKV) * D]
    part = lambda c, h, f: wide[:, c:c + h * f].view(B, 1, h, f).transpose(1, 2)
    q, k, v = part(cut[0], H, D), part(cut[1], HKV, D), part(cut[2], HKV, D)
    rk = part(cut[3], HG, R) if HG else None
    kc, vc = mk(B, HKV, 7, D), mk(B, 7, HKV, D).transpose(1, 2)
    rc = mk(B, HG, 7, R) if HG else None
    old = [None if t is None else t.clone() for t in (kc, vc, rc)]
    wq, wk = (1 + 0.2 * mk(D), 1 + 0.2 * mk(D)) if norm else (None, None)
    cos, sin = (mk(D).clamp(-1, 1), mk(D).clamp(-1, 1)) if rope else (None, None)
    at = lambda t: None if t is None else t[:, :, 4:5]
    ver = kc._version
    out = _capi.native().decode_rows(q, k, v, rk, at(kc), at(vc), at(rc), wq, 1e-6, wk, 1e-3,
                                     cos, sin)
    torch.cuda.synchronize()
    assert out is not None and out.shape == (B, H, D)
    assert kc._version > ver

    def ref(x, w, eps):
        x = x.double()
        if w is not None:
            x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()
        if cos is not None:
            h = torch.cat((-x[..., D // 2:], x[..., :D // 2]), -1)
            x = x * cos.double() + h * sin.double()
        return x

    # roundings to bf16, 2^-8 of the value each: the normalised x and its
    # partner before the rotation (|x cos| + |partner sin|), then the result
    for got, x, w, eps in ((out[:, :, None], q, wq, 1e-6), (at(kc), k, wk, 1e-3)):
        r = ref(x, w, eps)
        lim = torch.zeros_like(r)
        if norm:
            n = x.double()
            n = n * torch.rsqrt(n.square().mean(-1, keepdim=True) + eps) * w.double()
            part = torch.cat((n[..., D // 2:], n[..., :D // 2]), -1)
            lim += n.abs() if cos is None else (n * cos.double()).abs() + (part * sin.double()).abs()
        if rope:
            lim += r.abs()
        # (1 + 2^-6: the first roundings within the second, and the fp32 sums)
        assert ((got.double() - r).abs() <= 2 ** -8 * (1 + 2 ** -6) * lim).all()
    assert torch.equal(at(vc), v)
    if HG:
        assert torch.equal(at(rc), rk)
    for t, o in zip((kc, vc, rc), old):  # every other row as it was
        if t is not None:
            keep = [0, 1, 2, 3, 5, 6]
            assert torch.equal(t[:, :, keep], o[:, :, keep])


@pytest.mark.gpu
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("kw", [dict(), dict(use_qk_norm=False), dict(use_rope=False),
                                dict(n_kv_heads=2)], ids=str)
def test_module_step_against_torch_modules(gpu, bias, kw):
    from fna2_amd import attention_fna2 as A
    torch.manual_seed(0)
    m = A.NaylisAttention(512, 8, rel_rank=16, max_seq_len=64, decode_graph_bias=bias,
                          **kw).to(gpu).bfloat16().eval()
    assert m._use_fna2
    x = torch.randn(3, 1, 512, device=gpu).bfloat16()
    kv = kw.get("n_kv_heads", 8)

    def step(fused, cls=A.StaticKVCache):
        c = cls.empty(3, kv, 12, 64, 8 if bias else 0, 16, device=gpu)
        g = torch.Generator(device=gpu).manual_seed(1)
        rows = [torch.randn(3, h, 10, f, device=gpu, generator=g).bfloat16()
                for h, f in ((kv, 64), (kv, 64)) + (((8, 16),) if bias else ())]
        c.append(*rows)
        if not fused:
            m._decode_rows = lambda *a: None
        try:
            with torch.no_grad():
                y, _ = m(x, past_kv=c, use_kv_cache=True)
        finally:
            m.__dict__.pop("_decode_rows", None)
        assert c.length == 11
        return [y] + [t[:, :, 10] for t in (c.k, c.v, c.r_k) if t is not None]
    for a, b in zip(step(True), step(False)):
        # the torch chain rounds each of its about six steps to bf16
        assert (a.double() - b.double()).norm() <= 0.015 * b.double().norm()
    # a hooked norm is called as a module, a full cache raises as before
    if m.q_norm is not None:
        calls = []
        h = m.q_norm.register_forward_hook(lambda *a: calls.append(1))
        step(True)
        h.remove()
        assert calls
        h = torch.nn.modules.module.register_module_forward_pre_hook(
            lambda mod, a: calls.append(mod))
        step(True)
        h.remove()
        assert m.q_norm in calls
    # a cache of another class appends by its own method

    class Cache(A.StaticKVCache):
        n = 0

        def append(self, *rows):
            Cache.n += 1
            super().append(*rows)
    step(True, Cache)
    assert Cache.n == 2
    full = A.StaticKVCache.empty(3, kv, 4, 64, 8 if bias else 0, 16, device=gpu)
    full.length = 4
    with pytest.raises(ValueError, match="full"), torch.no_grad():
        m(x, past_kv=full, use_kv_cache=True)


@pytest.mark.gpu
@pytest.mark.parametrize("kw", [dict(), dict(use_qk_norm=False)], ids=str)
def test_step_under_autocast(gpu, kw):
    """Under autocast the norm's square and root run in fp32, and with them
    the rotary table: the step is the torch modules', and the row it appends
    is rotated by exact angles, as the prompt's rows are."""
    from fna2_amd import attention_fna2 as A
    torch.manual_seed(0)
    m = A.NaylisAttention(256, 4, rel_rank=16, max_seq_len=512, decode_graph_bias=True,
                          **kw).to(gpu).bfloat16().eval()
    x = torch.randn(2, 1, 256, device=gpu).bfloat16()
    n = 257

    def step(fused):
        g = torch.Generator(device=gpu).manual_seed(1)
        c = A.StaticKVCache.empty(2, 4, n + 1, 64, 4, 16, device=gpu)
        c.append(*(torch.randn(2, 4, n, f, device=gpu, generator=g).bfloat16() for f in (64, 64, 16)))
        if not fused:
            m._decode_rows = lambda *a: None
        try:
            with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
                y, _ = m(x, past_kv=c, use_kv_cache=True)
        finally:
            m.__dict__.pop("_decode_rows", None)
        return y, c.k[:, :, n]
    if kw:  # without the norm nothing is promoted: the bf16 table on both sides
        for a, b in zip(step(True), step(False)):
            assert (a.double() - b.double()).norm() <= 0.015 * b.double().norm()
        return
    (y, k), (y0, k0) = step(True), step(False)
    assert torch.equal(k, k0) and torch.equal(y, y0)
    with torch.no_grad():
        kk = m._project(x)[1].double()
        kk = kk * torch.rsqrt(kk.square().mean(-1, keepdim=True) + 1e-6) * m.k_norm.weight.double()
        ang = n * m.rope.inv_freq.double()
        c, s = ang.cos().repeat(2), ang.sin().repeat(2)
        h = torch.cat((-kk[..., 32:], kk[..., :32]), -1)
    assert (k.double() - (kk * c + h * s)[:, :, 0]).norm() <= 2 ** -7 * k.double().norm()


def test_rotary_table_is_left_alone():
    """A step that the torch modules take (here fp32 norm weights over bf16
    projections, CPU tensors) does not touch the rotary table: the table
    holds one dtype, and two callers of two dtypes would rebuild it each step."""
    from fna2_amd import attention_fna2 as A
    m = A.NaylisAttention(128, 2, rel_rank=16, max_seq_len=64).bfloat16().eval()
    m.q_norm.float()
    m.k_norm.float()
    c = A.StaticKVCache.empty(1, 2, 8, 64, 0, 16, device="cpu")
    c.append(torch.zeros(1, 2, 4, 64).bfloat16(), torch.zeros(1, 2, 4, 64).bfloat16())
    with torch.no_grad():
        q, k, v, _, _ = m._project(torch.randn(1, 1, 128).bfloat16())
        assert m._decode_rows(q, k, v, None, c) is None
    assert m.rope._cache_key is None and c.length == 4
