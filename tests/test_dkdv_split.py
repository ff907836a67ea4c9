"""dK/dV items in chunks (fna2_bwd_dkdv.hip with SPLIT, kv_reduce_kernel).

CPU: the chunks of an item cover its (head, query block) sequence once, and
the reduction reads exactly the dRk slots the chunks write (kv_chunks,
drk_slots in fna2_kernels.h restated).  GPU: gradients of shapes whose items
run in chunks against the oracle, and against the same call without the room
for chunks (the whole-item kernels): chunks that end inside a head, at heads'
ends, empty chunks, key tiles no query sees, ragged packs, cross lengths.
"""
import ctypes
import math

import pytest
import torch

from . import helpers as Hp

MIN_CHUNK = 4


def kv_chunks(blocks, log2):
    n = max(-(-blocks // (1 << log2)), MIN_CHUNK)
    return -(-blocks // n), n


@pytest.mark.parametrize("log2", [1, 2, 3, 4])
@pytest.mark.parametrize("group", [1, 2, 3, 8])
def test_chunks_cover_an_item_once(group, log2):
    for nqb in list(range(0, 40)) + [127, 512]:
        n, length = kv_chunks(group * nqb, log2)
        assert n <= 1 << log2
        seen, wrote, whole = [], {}, set()
        for s in range(n):  # the cursor's walk of a chunk
            first = s * length
            hi, at = divmod(first, nqb)
            left = min(group * nqb - first, length)
            while True:
                seg = min(nqb - at, left)
                assert seg > 0
                left -= seg
                seen += [(hi, at + i) for i in range(seg)]
                if seg == nqb:
                    whole.add(hi)
                else:
                    assert s + hi not in wrote, "two segments in one dRk slot"
                    wrote[s + hi] = hi
                    assert s + hi < group + (1 << log2) - 1
                if left == 0:
                    break
                hi, at = hi + 1, 0
        assert seen == [(h, q) for h in range(group) for q in range(nqb)]
        reads = {}
        for h in range(group if n > 1 else 0):  # kv_reduce_kernel
            c0, c1 = h * nqb // length, ((h + 1) * nqb - 1) // length + 1
            if c1 - c0 > 1:
                reads.update({c + h: h for c in range(c0, c1)})
                assert h not in whole
            else:
                assert h in whole
        if n > 1:
            assert reads == wrote
        else:
            assert not wrote


def _split_bytes(prob):
    from fna2_amd import _capi
    return int(_capi.lib().fna2_bwd_split_bytes(ctypes.byref(prob)))


def _problem(varlen, B, Sq, Sk, H, HKV, HG, D, R, causal, cu=None):
    import importlib
    F = importlib.import_module("fna2_amd.flash_naylis_attn")
    tq, tk = (Sq, Sk) if varlen else (0, 0)
    return F._problem(varlen, B, Sq, Sk, tq, tk, H, HKV, HG, D, R, causal, 0.1, cu, cu)


def test_split_rule():
    """Chunks where the items leave CUs idle, none where they fill them."""
    few = _split_bytes(_problem(False, 2, 1531, 1531, 16, 4, 12, 128, 24, True))
    assert few > 0
    # fp32 dK | dV of every chunk of every 128-key tile, at least two chunks
    assert few >= 2 * 2 * 12 * 4 * 2 * 128 * 2 * 128 * 4 // 2
    assert _split_bytes(_problem(False, 4, 2048, 2048, 16, 16, 16, 64, 16, True)) == 0
    assert _split_bytes(_problem(False, 1, 16384, 16384, 32, 32, 32, 128, 64, True)) == 0
    assert _split_bytes(_problem(False, 1, 64, 64, 8, 8, 8, 64, 32, True)) == 0
    assert _split_bytes(_problem(False, 2, 0, 128, 4, 4, 4, 64, 32, True)) == 0


DENSE = [  # B, Sq, Sk, H, HKV, HG, D, R, causal, fp16
    (1, 512, 512, 8, 4, 4, 64, 32, True, False),
    (1, 1000, 1000, 3, 1, 2, 64, 16, True, False),
    (1, 700, 700, 6, 2, 5, 64, 64, False, False),
    (1, 900, 900, 4, 2, 3, 128, 64, True, False),
    (2, 513, 513, 8, 2, 6, 128, 24, True, True),
    (1, 1025, 1025, 2, 2, 1, 64, 8, True, True),
    (1, 333, 1200, 4, 1, 4, 128, 32, True, False),   # key tiles no query sees
    (1, 1500, 70, 4, 4, 4, 128, 0, False, False),    # one key tile, no rank
]


def _run_dense(gpu, c, split):
    import importlib
    F = importlib.import_module("fna2_amd.flash_naylis_attn")
    B, Sq, Sk, H, HKV, HG, D, R, causal, fp16 = c
    ins = Hp.make_dense(B, H, Sq, D, HKV, HG if R else 0, R, seed=Sq + D + R, Sk=Sk)
    if fp16:
        ins = tuple(t if t is None or i in (3, 4, 5) else t.half() for i, t in enumerate(ins))
    q, k, v, rq, rk, gs, dout = (None if t is None else t.to(gpu) for t in ins)
    scale = 1 / math.sqrt(D)
    out, lse = F._fna2_forward(q, k, v, rq, rk, gs, scale, causal)
    lib = F._capi.lib()
    keep, native = lib.fna2_bwd_split_bytes, F._native_bwd
    try:
        if not split:  # the Python launcher, with a workspace that has no room for chunks
            lib.fna2_bwd_split_bytes = lambda p: 0
            F._native_bwd = lambda *a, **kw: None
        grads = F._fna2_backward(dout, q, k, v, rq, rk, gs, out, lse, scale, causal)
    finally:
        lib.fna2_bwd_split_bytes, F._native_bwd = keep, native
    torch.cuda.synchronize()
    return ins, scale, grads


@pytest.mark.gpu
@pytest.mark.parametrize("case", DENSE, ids=lambda c: "-".join(map(str, c)))
def test_dense_chunks(gpu, case):
    B, Sq, Sk, H, HKV, HG, D, R, causal, fp16 = case
    print(case, flush=True)
    assert _split_bytes(_problem(False, B, Sq, Sk, H, HKV, HG if R else 0, D, R, causal)) > 0
    ins, scale, got = _run_dense(gpu, case, True)
    _, _, whole = _run_dense(gpu, case, False)
    _, _, again = _run_dense(gpu, case, True)
    for a, b, c in zip(got, whole, again):
        if a is None:
            continue
        assert torch.equal(a, c), "not reproducible"
        # the same fp32 terms in another order, rounded once to 16 bits
        # (at most 2^-8 of a value on each side, and the same for most)
        assert Hp.rel_norm(a, b.double().cpu().numpy()) < 4e-3
    q, k, v, rq, rk, gs, dout = ins
    _, _, ref = Hp.oracle_fwd_bwd(q, k, v, rq, rk, gs, dout, scale, causal)
    Hp.check_grads(got[:5], ref[:5])


@pytest.mark.gpu
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("D,R", [(64, 16), (128, 32)])
def test_varlen_chunks(gpu, causal, D, R):
    """One long sequence beside short and empty ones, tokens outside every
    sequence, a vanilla head; every tile in chunks as long as it has blocks."""
    import importlib
    F = importlib.import_module("fna2_amd.flash_naylis_attn")
    lens, H, HKV, HG = [40, 0, 1300, 17, 129], 4, 2, 3
    q, k, v, rq, rk, gs, dout, cu, _ = Hp.make_varlen(lens + [9], H, D, HKV, HG, R, seed=D)
    cu = cu[:-1]
    dev = [t.to(gpu) for t in (q, k, v, rq, rk, gs, dout, cu)]
    dq, dk, dv, drq, drk, dgs, ddo, dcu = dev
    scale = 1 / math.sqrt(D)
    prob = F._problem(True, len(lens), 1300, 1300, q.shape[0], q.shape[0], H, HKV, HG, D, R,
                      causal, scale, dcu, dcu)
    assert _split_bytes(prob) > 0
    print("varlen chunks", D, R, causal, flush=True)
    out, lse = F._fna2_forward_varlen(dq, dk, dv, drq, drk, dgs, dcu, dcu, 1300, 1300, scale,
                                      causal)
    got = F._fna2_backward_varlen(ddo, dq, dk, dv, drq, drk, dgs, out, lse, dcu, dcu, 1300, 1300,
                                  scale, causal)
    torch.cuda.synchronize()
    n = sum(lens)
    ref_o, ref_l, ref = Hp.oracle_fwd_bwd(q, k, v, rq, rk, gs, dout, scale, causal, cu.numpy(),
                                          cu.numpy())
    for g, r in zip(got[:5], ref[:5]):
        assert not g[n:].any(), "rows outside every sequence"
        assert Hp.rel_norm(g[:n], r[:n]) < Hp.TOL_GRAD


@pytest.mark.gpu
@pytest.mark.parametrize("path", ["native", "python"])
def test_without_memory_for_chunks(gpu, monkeypatch, path):
    """Where the chunks' partials do not fit in memory the items run whole:
    the same gradients as with a workspace that has no room for chunks."""
    import importlib
    F = importlib.import_module("fna2_amd.flash_naylis_attn")
    S, H, D, room = 4096, 8, 128, 40 << 20
    prob = _problem(False, 1, S, S, H, 1, 0, D, 0, True)
    assert _split_bytes(prob) > room
    g = torch.Generator(device=gpu).manual_seed(5)
    q, k, v, dout = (torch.randn(1, h, S, D, device=gpu, generator=g).bfloat16()
                     for h in (H, 1, 1, H))
    args = (q, k, v, None, None, None)
    out, lse = F._fna2_forward(*args, 0.1, True)
    if path == "python":
        monkeypatch.setattr(F, "_native_bwd", lambda *a, **kw: None)
    # the gradients (10 MiB) and the other scratch fit in `room`
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(gpu).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved(gpu) + room) / total, gpu)
    try:
        got = F._fna2_backward(dout, *args, out, lse, 0.1, True)
        torch.cuda.synchronize()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, gpu)
    monkeypatch.setattr(F, "_native_bwd", lambda *a, **kw: None)
    monkeypatch.setattr(F._capi.lib(), "fna2_bwd_split_bytes", lambda p: 0)
    whole = F._fna2_backward(dout, *args, out, lse, 0.1, True)
    for a, b in zip(got[:3], whole[:3]):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("D,R", [(64, 16), (128, 32)])
def test_whole_items_after_the_chunks(gpu, causal, D, R):
    """A pack with more key tiles than the rule cuts: the longest in chunks,
    the last of the short ones whole, in one launch."""
    import importlib
    F = importlib.import_module("fna2_amd.flash_naylis_attn")
    lens, H, HKV, HG = [2000] + [33] * 29, 8, 1, 6
    total, N, bn = sum(lens), len(lens), 256 if D == 64 else 128
    q, k, v, rq, rk, gs, dout, cu, _ = Hp.make_varlen(lens, H, D, HKV, HG, R, seed=D)
    dev = [t.to(gpu) for t in (q, k, v, rq, rk, gs, dout, cu)]
    dq, dk, dv, drq, drk, dgs, ddo, dcu = dev
    scale = 1 / math.sqrt(D)
    prob = F._problem(True, N, 2000, 2000, total, total, H, HKV, HG, D, R, causal, scale, dcu, dcu)
    cut = max(N * -(-(total // N) // bn), -(-total // bn) + 8)
    assert cut < sum(-(-n // bn) for n in lens)
    # partials of `cut` tiles: dK | dV of 2^l chunks, dRk of 2^l + group - 1
    assert _split_bytes(prob) in [cut * bn * 4 * ((2 * D << l) + (H + (1 << l) - 1) * 32)
                                  for l in range(1, 5)]
    print("whole after chunks", D, R, causal, flush=True)
    out, lse = F._fna2_forward_varlen(dq, dk, dv, drq, drk, dgs, dcu, dcu, 2000, 2000, scale,
                                      causal)
    run = lambda: F._fna2_backward_varlen(ddo, dq, dk, dv, drq, drk, dgs, out, lse, dcu, dcu, 2000,
                                          2000, scale, causal)
    got, again = run(), run()
    lib = F._capi.lib()
    keep, native = lib.fna2_bwd_split_bytes, F._native_bwd
    try:
        lib.fna2_bwd_split_bytes, F._native_bwd = lambda p: 0, lambda *a, **kw: None
        whole = run()
    finally:
        lib.fna2_bwd_split_bytes, F._native_bwd = keep, native
    torch.cuda.synchronize()
    for a, b, c in zip(got, whole, again):
        assert torch.equal(a, c), "not reproducible"
        assert Hp.rel_norm(a, b.double().cpu().numpy()) < 4e-3  # (as in test_dense_chunks)
    for i in (1, 2):  # the whole items' keys: the last seven short sequences
        assert torch.equal(got[i][-33:], whole[i][-33:])
    _, _, ref = Hp.oracle_fwd_bwd(q, k, v, rq, rk, gs, dout, scale, causal, cu.numpy(), cu.numpy())
    Hp.check_grads(got[:5], ref[:5])


def test_split_rule_does_not_trust_max_seqlen():
    """A loose max_seqlen (the token count, none) does not cut the items of
    short sequences."""
    for hint in (0, 128, 768, 4096):
        p = _problem(True, 32, hint, hint, 8, 4, 8, 64, 16, True, None)
        p.total_q = p.total_k = 4096
        p.cu_seqlens_q = p.cu_seqlens_k = 1 << 20
        assert _split_bytes(p) == 0
    # one long sequence is known by its mean
    p = _problem(True, 2, 0, 0, 8, 4, 8, 64, 16, True, None)
    p.total_q = p.total_k = 4096
    p.cu_seqlens_q = p.cu_seqlens_k = 1 << 20
    assert _split_bytes(p) > 0


def test_equal_chunks_go_in_whole_rounds():
    """Without the mask the chunks are alike: 312 halves of 156 items are two
    rounds of 256 CUs, no shorter than the items whole."""
    assert _split_bytes(_problem(False, 3, 3209, 3209, 12, 4, 12, 64, 16, False)) == 0
    # 104 items: one round of halves
    halves = 2 * 13 * 4 * 256 * 4 * ((2 * 64 << 1) + (3 + (1 << 1) - 1) * 32)
    assert _split_bytes(_problem(False, 2, 3209, 3209, 12, 4, 12, 64, 16, False)) == halves


def test_token_count_as_max_seqlen_makes_no_rounds():
    """Lengths of 8000, 900, 700 and 617: 504 long items that 256 CUs share,
    not three rounds of them, whatever max_seqlen says; but one long sequence
    whose items do leave CUs idle is cut, and so is a pack of one sequence,
    whose items are alike."""
    def pack(total, n, hint, H, HKV, D, R):
        p = _problem(True, n, hint, hint, H, HKV, H if R else 0, D, R, False, None)
        p.total_q = p.total_k = total
        p.cu_seqlens_q = p.cu_seqlens_k = 1 << 20
        return _split_bytes(p)
    for hint in (0, 8000, 10217):
        assert pack(10217, 4, hint, 32, 8, 128, 64) == 0
    assert pack(10533, 4, 7083, 12, 4, 64, 0) > 0
    assert pack(4824, 1, 4824, 16, 8, 128, 16) > 0
