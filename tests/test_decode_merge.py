"""The decode's split rule for few units, and the merge of the splits at the
counts where its rounds and waves change (fna2_decode.hip merge_body)."""
import ctypes

import pytest
import torch

from fna2_amd import _capi


def _splits(B, H, HKV, HG, D, R, L, ragged=False):
    a = _capi.DecodeArgs()
    a.batch, a.heads, a.heads_kv, a.heads_graph = B, H, HKV, HG
    a.head_dim, a.rank, a.max_seqlen_k, a.softmax_scale = D, R, L, 0.1
    fake = 1 << 20
    for n in ("q", "r_q", "k_cache", "v_cache", "rk_cache", "out"):
        setattr(a, n, _capi.Tensor(fake, 1 << 20, 128, 1 << 14))
    a.graph_scale = fake
    a.seqlens_k = fake if ragged else None
    return _capi.lib().fna2_decode_num_splits(ctypes.byref(a))


@pytest.mark.parametrize("L,n", [(0, 1), (1, 1), (64, 1), (65, 1), (128, 1), (160, 5), (2048, 64),
                                 (4096, 64)])
def test_few_units_split_to_single_steps(L, n):
    """Once the chain of steps is longer than a second launch."""
    assert _splits(1, 8, 8, 0, 128, 0, L) == n


def test_many_units_keep_long_splits():
    assert _splits(64, 16, 16, 16, 128, 32, 4096) == 1
    assert _splits(16, 16, 16, 16, 128, 32, 2048) == 4
    assert _splits(64, 16, 16, 16, 128, 32, 128) == 1


@pytest.mark.parametrize("call,most", [
    # a few steps: a second launch costs more (measured whole / split, us)
    ((4, 4, 1, 0, 64, 0, 84, True), 1),         # 5.2 / 7.4
    ((87, 4, 1, 0, 64, 0, 84, True), 1),        # 5.6 / 7.9
    ((2, 8, 2, 8, 128, 16, 73, True), 1),       # 8.0 / 9.9
    ((13, 16, 16, 16, 64, 8, 116, True), 1),    # 7.9 / 9.1
    ((97, 32, 32, 0, 128, 0, 304, True), 1),    # 59 / 72 to 123
    # one round of the waves that fit, not a little more than one
    ((118, 4, 2, 4, 128, 8, 305, False), 4),    # 15.1 in four, 19.2 in five
    ((26, 32, 4, 32, 64, 16, 339, False), 6),   # 13.3 in six, 18.6 in eleven
    ((1, 32, 32, 32, 128, 32, 1239, False), 20),  # 11.3 in twenty, 15.6 in 39
    ((20, 32, 8, 0, 128, 0, 6000, False), 6),   # 90 in six, 104 in seven
])
def test_calls_not_split_further(call, most):
    assert 1 <= _splits(*call) <= most


@pytest.mark.parametrize("L", list(range(1, 400, 7)) + [1023, 4095, 131072, 2 ** 30])
@pytest.mark.parametrize("B,H,HKV,HG,D,R", [(1, 1, 1, 0, 64, 0), (3, 32, 1, 8, 64, 32),
                                            (300, 8, 8, 8, 128, 64), (2 ** 16, 32, 32, 0, 128, 0)])
def test_counts_are_in_range(B, H, HKV, HG, D, R, L):
    for ragged in (False, True):
        assert 1 <= _splits(B, H, HKV, HG, D, R, L, ragged) <= min(64, -(-L // 32))


def _one_step(a, b, absolute):
    """a and b: one output in different splits.  P's two parts and the fp32
    sums leave each at most 2^-13 of sum P |V| (`absolute`) from the value
    itself; the output's rounding then puts them at most one bf16 step apart."""
    a, b, s = a.double(), b.double(), absolute.double()
    return ((a - b).abs() <= 2 ** -7 * torch.maximum(a.abs(), b.abs()) + 2 ** -12 * s).all()


@pytest.mark.gpu
def test_workspace_sized_without_lengths(gpu):
    """A ragged call may split more than the even one; with the even call's
    workspace it splits as that does."""
    from fna2_amd.decode import decode_args, flash_naylis_decode
    g = torch.Generator().manual_seed(1)
    mk = lambda *s: torch.randn(*s, generator=g).bfloat16().to(gpu)
    B, H, L = 130, 8, 600
    q, k, v = mk(B, H, 64), mk(B, H, L, 64), mk(B, H, L, 64)
    seq = torch.tensor([(7 * i) % (L + 1) for i in range(B)], dtype=torch.int32, device=gpu)
    lib = _capi.lib()
    a, keep, out, _ = decode_args(q, k, v, cache_seqlens=seq)
    big = lib.fna2_decode_workspace_bytes(ctypes.byref(a))
    a.seqlens_k = None
    small = lib.fna2_decode_workspace_bytes(ctypes.byref(a))
    assert small < big
    a.seqlens_k = keep[-1].data_ptr()
    ws = torch.empty(big, dtype=torch.uint8, device=gpu)
    a.workspace = ws.data_ptr()
    outs = []
    for n in (big, small):
        a.workspace_bytes = n
        st = lib.fna2_decode(ctypes.byref(a), torch.cuda.current_stream(gpu).cuda_stream)
        assert st == 0
        torch.cuda.synchronize()
        outs.append(out.clone())
    assert _one_step(outs[0], outs[1], flash_naylis_decode(q, k, v.abs(), cache_seqlens=seq))


@pytest.mark.gpu
@pytest.mark.parametrize("D,R", [(64, 16), (128, 32)])
@pytest.mark.parametrize("n", [2, 7, 8, 9, 16, 17, 31, 32, 33, 63, 64])
def test_merge_of_n_splits(gpu, n, D, R):
    from fna2_amd.decode import flash_naylis_decode
    print(n, D, R, flush=True)
    B, H, HKV, HG, L = 3, 6, 2, 4, 64 * 32
    g = torch.Generator().manual_seed(n + D)
    mk = lambda *s, f=1.0: (torch.randn(*s, generator=g) * f).bfloat16().to(gpu)
    q, k, v = mk(B, H, D), mk(B, HKV, L, D), mk(B, HKV, L, D)
    rq, rk = mk(B, HG, R, f=R ** -0.5), mk(B, HG, L, R, f=R ** -0.5)
    gs = torch.ones(HG, device=gpu)
    seq = torch.tensor([L, 33, 0], dtype=torch.int32, device=gpu)  # splits with no rows
    run = lambda s, v=v: flash_naylis_decode(q, k, v, rq, rk, gs, cache_seqlens=seq, num_splits=s,
                                             return_lse=True)
    (o, l), (o1, l1) = run(n), run(1)
    torch.cuda.synchronize()
    # (the LSE is an fp32 sum)
    assert _one_step(o, o1, run(1, v.abs())[0])
    fin = torch.isfinite(l1)
    assert torch.equal(torch.isfinite(l), fin) and not fin[2].any()
    assert (l - l1)[fin].abs().max() < 1e-5
    assert not o[2].any()
    assert torch.equal(run(n)[0], o)


@pytest.mark.gpu
@pytest.mark.parametrize("splits", [1, 2, 7])
@pytest.mark.parametrize("D", [64, 128])
def test_error_is_the_outputs_rounding(gpu, D, splits):
    """The probabilities enter their product within 2^-14, so the error is
    the bf16 output's rounding: at most 2^-8 of each value, and 2^-8 / sqrt(3)
    x 0.68 in the norm for significands spread over [1, 2) (0.0015; P in bf16
    alone gave 0.0020 to 0.0022)."""
    from fna2_amd.decode import flash_naylis_decode
    g = torch.Generator().manual_seed(D + splits)
    q, k, v = (torch.randn(*s, generator=g).bfloat16() for s in
               ((3, 8, D), (3, 4, 1500, D), (3, 4, 1500, D)))
    s = q.double().view(3, 4, 2, D) @ k.double().transpose(2, 3) * D ** -0.5
    ref = (torch.softmax(s, -1) @ v.double()).view(3, 8, D)
    got = flash_naylis_decode(q.to(gpu), k.to(gpu), v.to(gpu), num_splits=splits).cpu().double()
    assert (got - ref).norm() <= (2 ** -9 + 2 ** -16) * ref.norm()
    scale = (torch.softmax(s, -1) @ v.double().abs()).view(3, 8, D)
    assert ((got - ref).abs() <= 2 ** -8 * ref.abs() + 2 ** -13 * scale).all()


@pytest.mark.gpu
@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("D,R", [(64, 0), (128, 32)])
def test_infinite_values(gpu, D, R, splits):
    """An infinite V gives an infinite output where its key has weight, as
    torch does, also at a split's maximum (P = 1, no second part) and where P
    rounds up to bf16; NaN stays in its feature."""
    from fna2_amd.decode import flash_naylis_decode
    g = torch.Generator().manual_seed(D + splits)
    B, H, HKV, L = 2, 4, 2, 200
    q, k, v = (torch.randn(*s, generator=g).bfloat16() for s in
               ((B, H, D), (B, HKV, L, D), (B, HKV, L, D)))
    bias = ()
    if R:
        bias = (torch.randn(B, H, R, generator=g).bfloat16() * R ** -0.5,
                torch.randn(B, H, L, R, generator=g).bfloat16(), torch.ones(H))
    s = (q.double().view(B, HKV, 2, D) @ k.double().transpose(2, 3)).view(B, H, L) * D ** -0.5
    if R:
        s += (bias[1].double() @ bias[0].double()[..., None])[..., 0]
    top = s[0, 0].argmax().item()
    inf = float("inf")
    v[0, 0, top, 3] = inf
    for j in range(8):  # eight keys' weights: rounded up, rounded down
        v[0, 1, 17 + 23 * j, 5 + j] = inf if j % 2 else -inf
    v[1, 0, 199, D - 1] = -inf
    v[1, 1, 40, 8], v[1, 1, 41, 8] = inf, -inf
    v[1, 1, 0, 9] = float("nan")
    ref = (torch.softmax(s, -1).view(B, HKV, 2, L) @ v.double()).view(B, H, D)
    got = flash_naylis_decode(*(t.to(gpu) for t in (q, k, v, *bias)), num_splits=splits).cpu()
    fin = torch.isfinite(ref)
    assert (~fin).sum() == 2 * (1 + 8 + 1 + 1 + 1)
    assert torch.equal(torch.isnan(got), torch.isnan(ref))
    assert torch.equal(got.double()[~fin & ~torch.isnan(ref)], ref[~fin & ~torch.isnan(ref)])
    assert (got.double() - ref)[fin].norm() <= 2 ** -8 * ref[fin].norm()
