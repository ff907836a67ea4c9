"""The rotary kernels where their tokens per wave, row passes and shared
angle table change: token counts around the rule's limits, heads that do not
fill a pass, head dims from 16 to 512 (a table wider than the wave), in the
16-bit types and fp32, with and without norms.  Compared with the formula in
fp64 (the forward without a norm in 16 bits rounds its table: compared with
itself on a longer pack instead)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _ref(x, w, cu, inv, eps):
    x = x.double()
    pos = torch.zeros(x.shape[0], dtype=torch.float64, device=x.device)
    inside = torch.zeros(x.shape[0], dtype=torch.bool, device=x.device)
    for a, b in zip(cu[:-1], cu[1:]):
        pos[a:b] = torch.arange(b - a, device=x.device, dtype=torch.float64)
        inside[a:b] = True
    h = x.shape[-1] // 2
    y = x if w is None else x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()
    # the kernel's angle is one fp32 product
    ang = (pos.float()[:, None] * inv).double()[:, None]
    r = torch.cat((y[..., :h] * ang.cos() - y[..., h:] * ang.sin(),
                   y[..., h:] * ang.cos() + y[..., :h] * ang.sin()), -1)
    return torch.where(inside[:, None, None], r, x)


CASES = [  # T, Hq, Hk, D
    (1, 1, 1, 64), (3, 3, 1, 128), (1024, 5, 2, 128), (1025, 4, 4, 64), (4096, 3, 3, 128),
    (4097, 2, 1, 128), (12288, 2, 2, 64), (12289, 1, 3, 64), (37, 9, 17, 16), (50, 2, 2, 512),
    (130, 0, 4, 256),
    # fp32, q and k in one pass: as many rows as it has, one more, one side empty
    (200, 8, 8, 64), (201, 9, 1, 64), (90, 4, 4, 128), (91, 1, 5, 128), (70, 1, 1, 512), (40, 0, 3, 128),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_norm_rope_forward_and_backward(gpu, case, dtype):
    from fna2_amd.rope import rope_varlen_bwd, rope_varlen_raw
    T, Hq, Hk, D = case
    print(case, dtype, flush=True)
    g = torch.Generator().manual_seed(T + D)
    mk = lambda h: torch.randn(T, h, D, generator=g).to(dtype).to(gpu)
    q, k, gq, gk = mk(Hq), mk(Hk), mk(Hq), mk(Hk)
    wq, wk = (1 + 0.2 * torch.randn(2, D, generator=g)).to(gpu)
    if T % 2 or Hq == 0:
        wq = None  # q rotated only, or no rows to have a gradient from
    inv = (1.0 / 10000 ** (torch.arange(0, D, 2).float() / D)).to(gpu)
    cu = [0, T // 3, T // 3, max(T - 2, T // 3)] if T > 3 else [0, T]
    dcu = torch.tensor(cu, dtype=torch.int32, device=gpu)
    eps = 1e-5
    qo, ko = rope_varlen_raw(q, k, dcu, inv, 1, wq, wk, eps)
    dq, dk, dwq, dwk = rope_varlen_bwd(gq, gk, q, k, dcu, inv, 1, wq, wk, eps)
    torch.cuda.synchronize()
    leaves = [t.double().requires_grad_(True) for t in (q, k)]
    ws = [None if w is None else w.double().requires_grad_(True) for w in (wq, wk)]
    # one rounding to the type after an fp32 chain of about ten operations
    tol = {torch.bfloat16: 2 ** -9, torch.float16: 2 ** -12, torch.float32: 2 ** -22}[dtype] * 2
    for got, x, w in ((qo, leaves[0], ws[0]), (ko, leaves[1], ws[1])):
        r = _ref(x, w, cu, inv, eps)
        assert (got.double() - r).norm() <= tol * r.norm() + 1e-12
    outs = [_ref(x, w, cu, inv, eps) for x, w in zip(leaves, ws)]
    wanted = leaves + [w for w in ws if w is not None]
    loss = sum((o * y.double()).sum() for o, y in zip(outs, (gq, gk)))
    ref = torch.autograd.grad(loss, wanted, allow_unused=True)
    got = [dq, dk] + [d for d, w in ((dwq, wq), (dwk, wk)) if w is not None]
    for i, (a, b) in enumerate(zip(got, ref)):
        # (the weight gradients are fp32 sums over the rows)
        lim = tol if i < 2 else 2e-6
        assert (a.double() - b).norm() <= lim * b.norm() + 1e-6 * (i >= 2), i
