"""The forward's and dQ's key groups (fna2_fwd.hip, fna2_bwd_dq.hip, NG > 1)
where their steps and tiles end: key counts around multiples of a round of
groups, a last query tile of one row, tiles whose groups have no key at all
(causal), cross lengths, vanilla heads, both types; against the oracle.  CPU:
which problems run in key groups."""
import ctypes
import importlib
import math

import pytest
import torch

from . import helpers as Hp


def _groups(varlen, B, Sq, Sk, H, HG, D, R, causal, total=0, dtype=torch.bfloat16):
    """(forward, dQ) key groups; varlen: Sq, Sk are the max_seqlen hints."""
    F = importlib.import_module("fna2_amd.flash_naylis_attn")
    p = F._problem(varlen, B, Sq, Sk, total, total, H, H, HG, D, R, causal, 0.1, dtype=dtype)
    p.cu_seqlens_q = p.cu_seqlens_k = 1 << 20
    return tuple(F._capi.lib().fna2_key_groups(ctypes.byref(p), b) for b in (0, 1))


@pytest.mark.parametrize("call,groups", [
    # dense: B, S, H, D, R, causal
    ((1, 512, 8, 64, 16, True), (1, 1)), ((1, 768, 8, 64, 16, True), (4, 3)),
    ((1, 768, 8, 64, 64, True), (3, 2)), ((1, 768, 8, 64, 16, False), (1, 3)),
    ((1, 1024, 8, 64, 0, False), (4, 3)), ((1, 511, 8, 128, 32, True), (1, 1)),
    ((1, 512, 8, 128, 32, True), (3, 1)), ((1, 1024, 8, 128, 0, True), (3, 2)),
    ((1, 768, 8, 128, 0, False), (3, 1)), ((1, 1024, 16, 128, 32, False), (3, 2)),
    ((1, 1024, 32, 128, 32, False), (3, 1)), ((1, 2048, 16, 128, 32, False), (3, 2)),
    # past 256 tiles: causal, and few (sequence, head) pairs
    ((1, 1280, 32, 64, 16, True), (4, 3)), ((10, 768, 8, 64, 16, True), (1, 1)),
    ((1, 1024, 40, 64, 16, True), (1, 1)), ((2, 1531, 16, 128, 24, True), (3, 2)),
    ((1, 1531, 37, 128, 24, True), (1, 1)), ((1, 2048, 32, 64, 0, True), (1, 3)),
    ((1, 4096, 16, 64, 0, True), (4, 3)), ((1, 1280, 32, 64, 16, False), (1, 1)),
    ((1, 4096, 17, 64, 16, True), (1, 1)),
])
def test_which_dense_problems(call, groups):
    B, S, H, D, R, causal = call
    for dt in (torch.bfloat16, torch.float16):
        assert _groups(False, B, S, S, H, H if R else 0, D, R, causal, dtype=dt) == groups


def test_which_packs():
    """A pack's keys are the mean length that some sequence must have: a loose
    max_seqlen (the token count, none) does not send short packs here."""
    for hint in (0, 400, 768, 4000, 1 << 20):
        assert _groups(True, 10, hint, hint, 8, 8, 64, 16, True, 4000) == (1, 1)
    for hint in (0, 1000, 4000):
        assert _groups(True, 4, hint, hint, 4, 4, 64, 16, True, 4000) == (4, 3)
    # a hint below the mean: tokens outside every sequence
    assert _groups(True, 4, 500, 500, 4, 4, 64, 16, True, 4000) == (1, 1)
    assert _groups(True, 0, 0, 0, 8, 8, 64, 16, True, 4000)[0] >= 1


CASES = [  # B, Sq, Sk, H, HKV, HG, D, R, causal, fp16
    (1, 768, 768, 2, 1, 1, 64, 16, True, False),
    (1, 769, 769, 2, 2, 2, 64, 32, True, True),
    (1, 1000, 1000, 1, 1, 1, 64, 64, False, False),
    (1, 129, 1025, 2, 1, 0, 64, 0, False, False),
    (1, 33, 2049, 3, 3, 2, 64, 8, False, True),
    (1, 512, 512, 2, 2, 2, 128, 32, True, False),
    (1, 801, 801, 2, 1, 1, 128, 24, True, True),
    (2, 770, 770, 1, 1, 1, 128, 64, True, False),
    (1, 64, 833, 2, 2, 2, 128, 64, False, False),
    (1, 1100, 800, 2, 2, 1, 128, 16, True, False),
    (1, 1030, 1030, 2, 1, 1, 128, 24, True, True),
    (1, 1100, 1100, 1, 1, 1, 128, 64, True, False),
    (1, 129, 1025, 2, 1, 0, 128, 0, False, False),
    (1, 1025, 1025, 1, 1, 0, 128, 0, True, True),
    (1, 200, 1100, 2, 2, 2, 128, 32, False, False),
    (1, 130, 1100, 2, 2, 1, 64, 64, False, True),
    (1, 1200, 1400, 1, 1, 1, 64, 32, True, False),
]


def test_every_kernel_is_reached():
    """The dense cases below run every key-group kernel: D, rank tile (and
    the forward's R <= 16 at d = 64), bf16; fp16 for each D."""
    fwd, dq = set(), set()
    for B, Sq, Sk, H, HKV, HG, D, R, causal, fp16 in CASES:
        g = _groups(False, B, Sq, Sk, H, HG, D, R, causal)
        rpl = 0 if HG == 0 else 16 if R <= 16 and D == 64 else 32 if R <= 32 else 64
        if g[0] > 1:
            fwd |= {(D, rpl), (D, fp16)}
        if g[1] > 1:
            dq |= {(D, min(max(rpl, 32), 64) if rpl else 0), (D, fp16)}
    assert fwd >= {(64, 0), (64, 16), (64, 32), (64, 64), (128, 0), (128, 32), (128, 64)}
    assert dq >= {(64, 0), (64, 32), (64, 64), (128, 0), (128, 32), (128, 64)}
    assert fwd & dq >= {(D, t) for D in (64, 128) for t in (True, False)}


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_dense(gpu, case):
    F = importlib.import_module("fna2_amd.flash_naylis_attn")
    B, Sq, Sk, H, HKV, HG, D, R, causal, fp16 = case
    print(case, flush=True)
    ins = Hp.make_dense(B, H, Sq, D, HKV, HG, R, seed=Sq + Sk + D, Sk=Sk)
    if fp16:
        ins = tuple(t if t is None or i in (3, 4, 5) else t.half() for i, t in enumerate(ins))
    q, k, v, rq, rk, gs, dout = ins
    d = [None if t is None else t.to(gpu) for t in ins]
    scale = 1 / math.sqrt(D)
    out, lse = F._fna2_forward(*d[:6], scale, causal)
    grads = F._fna2_backward(d[6], *d[:6], out, lse, scale, causal)
    again = F._fna2_forward(*d[:6], scale, causal)
    torch.cuda.synchronize()
    assert torch.equal(out, again[0]) and torch.equal(lse, again[1])
    ref_o, ref_l, ref_g = Hp.oracle_fwd_bwd(q, k, v, rq, rk, gs, dout, scale, causal)
    Hp.check_out(out, lse, ref_o, ref_l)
    Hp.check_grads(grads[:5], ref_g[:5])


@pytest.mark.gpu
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("lens", [[900, 0, 31, 260], [2100, 17, 1000]], ids=str)
def test_varlen(gpu, causal, lens):
    """The second pack runs in key groups, its short sequences with them."""
    F = importlib.import_module("fna2_amd.flash_naylis_attn")
    H, D, R, m = 2, 128, 32, max(lens)
    assert (_groups(True, len(lens), m, m, H, H, D, R, causal, sum(lens)) == (3, 2)) == (m > 900)
    q, k, v, rq, rk, gs, dout, cu, _ = Hp.make_varlen(lens, H, D, 1, H, R, seed=3)
    d = [t.to(gpu) for t in (q, k, v, rq, rk, gs)]
    c, scale = cu.to(gpu), 1 / math.sqrt(D)
    print("varlen", causal, flush=True)
    out, lse = F._fna2_forward_varlen(*d, c, c, m, m, scale, causal)
    grads = F._fna2_backward_varlen(dout.to(gpu), *d, out, lse, c, c, m, m, scale, causal)
    torch.cuda.synchronize()
    ref_o, ref_l, ref_g = Hp.oracle_fwd_bwd(q, k, v, rq, rk, gs, dout, scale, causal, cu.numpy(),
                                            cu.numpy())
    Hp.check_out(out, lse, ref_o, ref_l)
    Hp.check_grads(grads[:5], ref_g[:5])
