"""The native launch path (csrc/fna2_torch.cpp) against the Python launchers:
the same call through both gives the same bits, and calls it does not take
(layouts to copy, dtypes to convert, errors to raise) go on as before."""
import importlib

import pytest
import torch

from . import helpers as Hp

F = importlib.import_module("fna2_amd.flash_naylis_attn")


@pytest.fixture
def native():
    from fna2_amd import _capi
    return _capi.native()


def test_cpu_tensors_are_left_to_the_python_launchers(native):
    t = torch.zeros(1, 2, 16, 64, dtype=torch.bfloat16)
    args = (t, t, t, None, None, None, 0.1, True, None, None, 0, 0, None, False, False)
    assert native.attn_fwd(*args) is None
    assert native.decode(t[:, :, 0], t, t, None, None, None, 0.1, None, 0) is None
    with pytest.raises(AssertionError, match="GPU tensor"):
        F._fna2_forward(t, t, t, None, None, None, 0.1, True)


def test_without_the_binding_the_python_launchers_run(monkeypatch):
    """A tree with the library and no (or another torch's) binding: one
    warning, and every entry point goes on through its Python launcher."""
    import types
    import warnings

    from fna2_amd import _capi

    def missing(*a):
        raise ImportError("undefined symbol")
    monkeypatch.setattr("importlib.import_module", missing)
    monkeypatch.setattr(_capi, "_native", None)
    monkeypatch.setattr(_capi, "_native_missing", False)
    t = types.SimpleNamespace(is_cuda=True)
    with pytest.warns(RuntimeWarning, match="does not load.*Python launchers"):
        assert F._native_fwd(t, t, t, None, None, None, 0.1, True) is None
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert F._native_bwd(t, t, t, t, None, None, None, t, t, 0.1, True) is None
        assert _capi.native_or_none() is None
    with pytest.raises(RuntimeError, match="build it"):
        _capi.native()


@pytest.mark.gpu
def test_without_the_binding_every_entry_point(gpu, monkeypatch):
    from fna2_amd import _capi, attention_fna2 as A
    torch.manual_seed(0)
    m = A.NaylisAttention(256, 4, rel_rank=16, max_seq_len=64, decode_graph_bias=True)
    m = m.to(gpu).bfloat16().eval()
    x, row = (torch.randn(2, s, 256, device=gpu).bfloat16() for s in (9, 1))

    def calls():
        c = A.StaticKVCache.empty(2, 4, 12, 64, 4, 16, device=gpu)
        with torch.no_grad():
            y, _ = m(x, past_kv=c, use_kv_cache=True)
            z, _ = m(row, past_kv=c, use_kv_cache=True)
        w, _ = m(x)
        return (y, z, *torch.autograd.grad(w.sum(), list(m.parameters())))
    a = calls()
    monkeypatch.setattr(_capi, "_native", None)
    monkeypatch.setattr(_capi, "_native_missing", True)
    b = calls()
    for i, (p, q) in enumerate(zip(a, b)):
        # (the decode step's rows then come from the torch modules)
        assert torch.equal(p, q) if i != 1 else Hp.rel_norm(p, q.double().cpu().numpy()) < 0.015


CALLS = [  # dense or lengths, H, HKV, HG, D, R, causal, fp16
    ((2, 130), 8, 4, 6, 64, 24, True, False),
    ((1, 65), 4, 4, 0, 128, 0, False, False),
    ((3, 200), 6, 2, 6, 128, 64, True, True),
    ([33, 0, 257, 1], 4, 2, 3, 64, 16, True, False),
    ([129, 40], 8, 8, 8, 128, 32, False, True),
]


def _both(fn, names):
    """fn through the native path and, with it off, through the Python one."""
    a = fn()
    keep = {n: getattr(F, n) for n in names}
    try:
        for n in names:
            setattr(F, n, lambda *x, **k: None)
        b = fn()
    finally:
        for n, f in keep.items():
            setattr(F, n, f)
    return a, b


@pytest.mark.gpu
@pytest.mark.parametrize("strided", [False, True])
@pytest.mark.parametrize("call", CALLS, ids=str)
def test_attention_bits(gpu, call, strided):
    shape, H, HKV, HG, D, R, causal, fp16 = call
    packed = isinstance(shape, list)
    if packed:
        *ins, cu, _ = Hp.make_varlen(shape, H, D, HKV, HG, R, seed=7)
        cu = cu.to(gpu)
        kw = dict(cu_seqlens_q=cu, cu_seqlens_k=cu, max_seqlen_q=max(shape),
                  max_seqlen_k=max(shape))
    else:
        B, S = shape
        ins = Hp.make_dense(B, H, S, D, HKV, HG, R, seed=7, layout="bshd" if strided else "bhsd")
        kw = {}
    ins = [t if t is None else t.to(gpu) for t in ins]
    if fp16:
        ins = [t if t is None or i in (3, 4, 5) else t.half() for i, t in enumerate(ins)]
    if strided and packed:  # rows of a wider buffer
        wide = [None if t is None or t.dim() < 2 else
                torch.zeros(t.shape[0], t.shape[1] + 1, t.shape[2], dtype=t.dtype, device=gpu)
                for t in ins]
        for i, w in enumerate(wide):
            if w is not None:
                w[:, :ins[i].shape[1]] = ins[i]
                ins[i] = w[:, :ins[i].shape[1]]
    *x, dout = ins
    leaves = [t.detach().requires_grad_(True) for t in x if t is not None]

    def run():
        it = iter(leaves)
        a = [None if t is None else next(it) for t in x]
        out = F.flash_naylis_attn(*a, is_causal=causal, **kw)
        return (out, *torch.autograd.grad(out, leaves, dout))
    assert F._native_fwd(*x, D ** -0.5, causal, **(dict(cu_q=cu, cu_k=cu) if packed else {})) \
        is not None, "this call belongs to the native path"
    a, b = _both(run, ["_native_fwd"])
    c, d = _both(run, ["_native_bwd"])
    for p, q, r, s in zip(a, b, c, d):
        assert p.stride() == q.stride() == r.stride() == s.stride()
        assert torch.equal(p, q) and torch.equal(p, r)
    # without chunks (the Python launcher gives them room too): the same
    for p, s in zip(a, d):
        assert torch.equal(p, s)


def _through_python(fn, monkeypatch):
    """fn as if the binding were not there."""
    from fna2_amd import _capi
    with monkeypatch.context() as m:
        m.setattr(_capi, "native_or_none", lambda: None)
        return fn()


def _same(a, b):
    for x, y in zip(a, b):
        assert (x is None) == (y is None)
        assert x is None or (x.stride() == y.stride() and torch.equal(x, y))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=str)
@pytest.mark.parametrize("D,H,HKV,norms", [(64, 8, 2, "qk"), (128, 3, 3, "q"), (128, 4, 1, "")])
def test_rope_bits(gpu, native, monkeypatch, dtype, D, H, HKV, norms):
    """The rotation and its backward, into new tensors and into slices of a
    wider one, with rows outside every sequence."""
    from fna2_amd import rope as Ro
    g = torch.Generator(device=gpu).manual_seed(D + H)
    T, cu = 201, torch.tensor([3, 70, 70, 195], dtype=torch.int32, device=gpu)
    mk = lambda *s: torch.randn(*s, generator=g, device=gpu).to(dtype)
    wide = mk(T, H + HKV, D)
    q, k = wide[:, :H], wide[:, H:]
    dq, dk = mk(T, H, D), mk(T, HKV, D)
    inv = 1.0 / 10000 ** (torch.arange(0, D, 2, device=gpu) / D)
    nq = 1 + 0.2 * mk(D) if "q" in norms else None
    nk = 1 + 0.2 * mk(D) if "k" in norms else None
    assert native.rope_fwd(q, k, cu, inv, 1, nq, nk, 1e-6) is not None
    for sign in (1, -1):
        fwd = lambda: Ro.rope_varlen_raw(q, k, cu, inv, sign, nq, nk, 1e-6)
        _same(fwd(), _through_python(fwd, monkeypatch))
    slabs = []

    def bwd(given=False):
        to = {}
        if given:
            slabs.append(torch.zeros(T, H + HKV + 1, D, device=gpu, dtype=dtype))
            to = dict(dq=slabs[-1][:, :H], dk=slabs[-1][:, H:H + HKV])
        return Ro.rope_varlen_bwd(dq, dk, q, k, cu, inv, 1, nq, nk, 1e-6, **to)
    one = bwd()
    _same(one, _through_python(bwd, monkeypatch))
    given = lambda: bwd(True)
    two = given()
    _same(two, _through_python(given, monkeypatch))
    assert torch.equal(slabs[0], slabs[1]) and not slabs[0][:, -1].any()
    for x, y in zip(one, two):
        assert x is None or torch.equal(x, y)


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,HKV,HG,D,R,L", [(3, 8, 2, 6, 64, 24, 700), (2, 4, 4, 0, 128, 0, 33),
                                               (5, 8, 1, 8, 128, 16, 1000)])
def test_decode_bits(gpu, native, monkeypatch, B, H, HKV, HG, D, R, L):
    """The decode: all rows or ragged ones, a cache in either order, q as
    [B, H, D] or [B, H, 1, D], graph_scale in fp32 or bf16, split or whole."""
    from fna2_amd.decode import flash_naylis_decode
    g = torch.Generator(device=gpu).manual_seed(B + L)
    mk = lambda *s: torch.randn(*s, generator=g, device=gpu).bfloat16()
    q, k, v = mk(B, 1, H, D).transpose(1, 2), mk(B, L, HKV, D).transpose(1, 2), mk(B, HKV, L, D)
    rq, rk = (mk(B, HG, 1, R), mk(B, HG, L, R)) if HG else (None, None)
    gs = 1 + 0.5 * mk(HG) if HG else None
    seq = torch.tensor([(17 + 211 * i) % (L + 1) for i in range(B)], dtype=torch.int32, device=gpu)
    row = lambda t, flat: t if t is None or not flat else t[:, :, 0]
    for flat in (True, False):
        for lens in (None, seq):
            for scale in (gs, gs if gs is None else gs.float()):
                for n in (0, 1, 3):
                    run = lambda: flash_naylis_decode(row(q, flat), k, v, row(rq, flat), rk, scale,
                                                      cache_seqlens=lens, num_splits=n,
                                                      return_lse=True)
                    _same(run(), _through_python(run, monkeypatch))
    assert native.decode(q, k, v, rq, rk, gs, 0.1, seq, 0) is not None


@pytest.mark.gpu
@pytest.mark.parametrize("path", ["native", "python"])
def test_calls_run_on_the_current_stream(gpu, native, monkeypatch, path):
    """Every entry point on a stream of its own: its inputs are written there
    behind a wait of some milliseconds, so a launch on any other stream would
    read the zeros that they held before."""
    from fna2_amd import _capi, attention_fna2 as A, decode as De, rope as Ro
    if path == "python":
        monkeypatch.setattr(_capi, "native_or_none", lambda: None)
    torch.manual_seed(0)
    H, HKV, D, R, S = 4, 2, 64, 16, 300
    rnd = lambda *s: torch.randn(*s, device=gpu).bfloat16()
    dense = [rnd(2, h, S, f) for h, f in ((H, D), (HKV, D), (HKV, D), (H, R), (H, R))]
    gs, dout = torch.ones(H, device=gpu), rnd(2, H, S, D)
    pack = [t.transpose(1, 2).reshape(2 * S, *t.shape[1:2], t.shape[3]) for t in dense]
    pdout = dout.transpose(1, 2).reshape(2 * S, H, D)
    cu = torch.tensor([0, S, 2 * S], dtype=torch.int32, device=gpu)
    inv, w = torch.ones(D // 2, device=gpu), 1 + 0.1 * rnd(D)
    m = A.NaylisAttention(256, H, rel_rank=R, max_seq_len=64).to(gpu).bfloat16().eval()
    x = rnd(2, 1, 256)

    def train(*a):
        leaves = [t.detach().requires_grad_(True) for t in a[:-1]]
        out = F.flash_naylis_attn(*leaves, is_causal=True)
        return (out, *torch.autograd.grad(out, leaves, a[-1]))

    def fwd_bwd_varlen(q, k, v, rq, rk, g, do):
        out, lse = F._fna2_forward_varlen(q, k, v, rq, rk, g, cu, cu, S, S, 0.125, True)
        return (out, lse, *F._fna2_backward_varlen(do, q, k, v, rq, rk, g, out, lse, cu, cu, S, S,
                                                   0.125, True))

    def step(row, k, v):
        c = A.StaticKVCache.empty(2, H, 8, D, device=gpu)
        with torch.no_grad():
            c.append(k, v)
            y, _ = m(row, past_kv=c, use_kv_cache=True)
        return y, c.k[:, :, :4], c.v[:, :, :4]
    calls = [
        ("train", train, (*dense, gs, dout)),
        ("varlen", fwd_bwd_varlen, (*pack, gs, pdout)),
        ("decode", lambda q, *a: De.flash_naylis_decode(q, *a, return_lse=True),
         (dense[0][:, :, 0], dense[1], dense[2], dense[3][:, :, 0], dense[4], gs)),
        ("rope", lambda q, k, a, b: Ro.rope_varlen_raw(q, k, cu, inv, 1, a, b, 1e-6),
         (pack[0], pack[1], w, w)),
        ("rope_bwd", lambda *a: Ro.rope_varlen_bwd(*a[:4], cu, inv, 1, *a[4:], 1e-6),
         (pdout, pack[1], pack[0], pack[1], w, w)),
        ("step", step, (x, rnd(2, H, 3, D), rnd(2, H, 3, D))),
    ]
    side = torch.cuda.Stream()
    for name, fn, args in calls:
        print(path, name, flush=True)
        ref = fn(*args)
        bufs = [torch.zeros_like(t) for t in args]
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            torch.cuda._sleep(5_000_000)
            for b, t in zip(bufs, args):
                b.copy_(t)
            got = fn(*bufs)
            waiting = not side.query()
        side.synchronize()
        assert waiting or path == "python", "the call waited for its stream"
        _same(got, ref)


@pytest.mark.gpu
def test_calls_left_to_the_python_launcher(gpu):
    q, k, v, rq, rk, gs, dout = [t.to(gpu) for t in Hp.make_dense(1, 4, 64, 64, 4, 4, 16)]
    s = 0.125
    ref, _ = F._fna2_forward(q, k, v, rq, rk, gs, s, True)
    # a feature stride of two: copied; graph_scale in bf16: converted
    wide = torch.zeros(*q.shape[:-1], 128, dtype=q.dtype, device=gpu)
    wide[..., ::2] = q
    assert F._native_fwd(wide[..., ::2], k, v, rq, rk, gs, s, True) is None
    assert torch.equal(F._fna2_forward(wide[..., ::2], k, v, rq, rk, gs, s, True)[0], ref)
    g16 = gs.bfloat16()
    assert F._native_fwd(q, k, v, rq, rk, g16, s, True) is None
    F._fna2_forward(q, k, v, rq, rk, g16, s, True)
    with pytest.raises(AssertionError, match="multiple of 8"):
        F._fna2_forward(q, k, v, rq[..., :12].contiguous(), rk[..., :12].contiguous(), gs, s, True)
    with pytest.raises(AssertionError, match="dtype"):
        F._fna2_forward(q, k.half(), v, rq, rk, gs, s, True)
    with pytest.raises(AssertionError, match="FNA2_E_SCALE"):
        F._fna2_forward(q, k, v, rq, rk, gs, float("nan"), True)


@pytest.mark.gpu
def test_numbers_of_other_types(gpu):
    """The numbers that the Python launchers convert: any real or integral
    object, also a float that holds a count."""
    from fna2_amd.decode import flash_naylis_decode
    q, k, v, rq, rk, gs, dout = [t.to(gpu) for t in Hp.make_dense(1, 4, 64, 64, 4, 4, 16)]
    ref = flash_naylis_decode(q[:, :, 0], k, v, softmax_scale=0.125, num_splits=2)
    got = flash_naylis_decode(q[:, :, 0], k, v, softmax_scale=torch.tensor(0.125), num_splits=2.0)
    assert torch.equal(got, ref)
    x = [t[0].transpose(0, 1).contiguous() for t in (q, k, v, rq, rk)]
    cu = torch.tensor([0, 40, 64], dtype=torch.int32, device=gpu)
    ref = F._fna2_forward_varlen(*x, gs, cu, cu, 40, 40, 0.125, True)
    got = F._fna2_forward_varlen(*x, gs, cu, cu, 40.0, torch.tensor(40), torch.tensor(0.125), 1)
    assert torch.equal(got[0], ref[0]) and torch.equal(got[1], ref[1])


@pytest.mark.gpu
def test_failed_launch_is_raised_not_repeated(gpu, native):
    """FNA2_E_LAUNCH may come after other kernels of the call were queued:
    it is raised, and no Python launcher or torch module runs the call again."""
    import ctypes

    from fna2_amd import _capi, attention_fna2 as A, decode as De, rope as Ro
    q, k, v, rq, rk, gs, dout = [t.to(gpu) for t in Hp.make_dense(1, 4, 64, 64, 4, 4, 16)]
    out, lse = F._fna2_forward(q, k, v, rq, rk, gs, 0.125, True)
    x = q[0].transpose(0, 1).contiguous()
    cu = torch.tensor([0, 64], dtype=torch.int32, device=gpu)
    inv = torch.ones(32, device=gpu)
    m = A.NaylisAttention(256, 4, rel_rank=16, max_seq_len=64).to(gpu).bfloat16().eval()
    cache = A.StaticKVCache.empty(1, 4, 8, 64, device=gpu)
    cache.length = 3
    row = torch.zeros(1, 1, 256, device=gpu).bfloat16()
    step = torch.no_grad()(lambda: m(row, past_kv=cache, use_kv_cache=True))
    calls = [("fna2_fwd", lambda: F._fna2_forward(q, k, v, rq, rk, gs, 0.125, True)),
             ("fna2_bwd", lambda: F._fna2_backward(dout, q, k, v, rq, rk, gs, out, lse, 0.125, True)),
             ("fna2_decode", lambda: De.flash_naylis_decode(q[:, :, 0], k, v)),
             ("fna2_decode_rows", step),
             ("fna2_rope_varlen", lambda: Ro.rope_varlen_raw(x, x, cu, inv)),
             ("fna2_rope_bwd", lambda: Ro.rope_varlen_bwd(x, x, x, x, cu, inv))]
    n = [0]

    @ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p)
    def fails(args, stream):
        n[0] += 1
        return -10
    good = _capi._addresses(_capi.lib())
    for name, call in calls:
        print(name, flush=True)
        native.bind({**good, name: ctypes.cast(fails, ctypes.c_void_p).value}, _capi.FNA2Error)
        try:
            n[0] = 0
            with pytest.raises(_capi.FNA2Error, match=f"{name}: FNA2_E_LAUNCH"):
                call()
            assert n[0] == 1
        finally:
            native.bind(good, _capi.FNA2Error)
        call()
    assert cache.length == 4
