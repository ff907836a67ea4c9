"""The forward's and dQ's key groups (fna2_fwd.hip, fna2_bwd_dq.hip, NG > 1)
where their steps and tiles end: key counts around multiples of a round of
groups, a last query tile of one row, tiles whose groups have no key at all
(causal), cross lengths, vanilla heads, both types; against the oracle."""
import importlib
import math

import pytest
import torch

from . import helpers as Hp

pytestmark = pytest.mark.gpu

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
]


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


@pytest.mark.parametrize("causal", [True, False])
def test_varlen(gpu, causal):
    F = importlib.import_module("fna2_amd.flash_naylis_attn")
    lens, H, D, R = [900, 0, 31, 260], 2, 128, 32
    q, k, v, rq, rk, gs, dout, cu, _ = Hp.make_varlen(lens, H, D, 1, H, R, seed=3)
    d = [t.to(gpu) for t in (q, k, v, rq, rk, gs)]
    c, scale = cu.to(gpu), 1 / math.sqrt(D)
    print("varlen", causal, flush=True)
    out, lse = F._fna2_forward_varlen(*d, c, c, 900, 900, scale, causal)
    grads = F._fna2_backward_varlen(dout.to(gpu), *d, out, lse, c, c, 900, 900, scale, causal)
    torch.cuda.synchronize()
    ref_o, ref_l, ref_g = Hp.oracle_fwd_bwd(q, k, v, rq, rk, gs, dout, scale, causal, cu.numpy(),
                                            cu.numpy())
    Hp.check_out(out, lse, ref_o, ref_l)
    Hp.check_grads(grads[:5], ref_g[:5])
