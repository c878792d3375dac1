"""fp32 inputs at head dims 64 / 128, whose products run as split bf16 products
on the matrix core: accuracy against fp64, exact behaviour under power-of-two
scales (every part of a split scales with its value), and infinities and NaN,
which must come out where fp32 arithmetic puts them."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(autouse=True)
def _gpu_only():
    if not torch.cuda.is_available():
        pytest.skip("needs an MI355X")


def _inputs(be, D, H, nb, topk, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    q, k, v, do = (torch.randn(1, H, be * nb, D, generator=g, device=DEV) for _ in range(4))
    sel = torch.stack([torch.randperm(nb, generator=torch.Generator().manual_seed(i))[:topk]
                       for i in range(H * nb)]).view(1, H, nb, topk).int().to(DEV)
    # block sizes at the edges of a 32-key chunk
    vbs = torch.tensor([[be, 1, 31, 32, 33, be - 1][i % 6] for i in range(nb)],
                       dtype=torch.int32, device=DEV)
    return q, k, v, do, sel, vbs


def _run(q, k, v, do, sel, vbs, be):
    from vsa_mi355x import mi355x as M
    leaves = [x.clone().requires_grad_() for x in (q, k, v)]
    out = M.mi355x_sparse_attention(*leaves, sel, vbs, block_size=(1, 1, be))
    return [out.detach(), *torch.autograd.grad(out, leaves, do)]


def _fp64(q, k, v, do, sel, vbs, be):
    """The same by masked dense attention in fp64, with autograd."""
    H, S, D = q.shape[1:]
    nb = S // be
    leaves = [x[0].double().requires_grad_() for x in (q, k, v)]
    on = torch.zeros(H, nb, nb, dtype=torch.bool, device=DEV).scatter_(-1, sel[0].long(), True)
    ok = (torch.arange(be, device=DEV) < vbs[:, None]).reshape(-1)
    mask = on.repeat_interleave(be, 1).repeat_interleave(be, 2) & ok
    s = torch.matmul(leaves[0], leaves[1].transpose(1, 2).contiguous()) / math.sqrt(D)
    p = torch.softmax(s.masked_fill(~mask, -math.inf), -1)
    out = torch.matmul(p, leaves[2])
    return [x[None] for x in (out.detach(), *torch.autograd.grad(out, leaves, do[0].double()))]


@pytest.mark.parametrize("be,D,nb,topk", [(64, 64, 12, 3), (64, 128, 9, 1), (128, 64, 7, 7),
                                          (128, 128, 8, 3), (256, 64, 6, 2), (256, 128, 7, 4)])
def test_against_fp64(be, D, nb, topk):
    x = _inputs(be, D, 2, nb, topk, be + D)
    # a score of magnitude up to 16 (log2 units) carries 2^-21 of rounding, so a
    # weight 2^-21 ln 2 = 3.3e-7; the products and sums add a few 2^-24 each
    for name, a, e in zip(("out", "dq", "dk", "dv"), _run(*x, be), _fp64(*x, be)):
        rel = ((a.double() - e).norm() / e.norm()).item()
        print(f"  be={be} D={D} {name}: rel-L2 {rel:.2e}", flush=True)
        assert rel <= 2e-6, (name, rel)


@pytest.mark.parametrize("be,D", [(64, 64), (256, 128)])
def test_power_of_two_scales_are_exact(be, D):
    q, k, v, do, sel, vbs = _inputs(be, D, 2, 6, 3, 5)
    ref = _run(q, k, v, do, sel, vbs, be)
    a, b, c = 2.0 ** 40, 2.0 ** -60, 2.0 ** 50
    got = _run(q * a, k / a, v * b, do * c, sel, vbs, be)
    for name, x, y, s in zip(("out", "dq", "dk", "dv"), got, ref, (b, b * c / a, b * c * a, c)):
        assert torch.equal(x, y * s), name


@pytest.mark.parametrize("be,D", [(64, 128), (128, 64), (256, 128)])
def test_infinities_and_nan(be, D):
    q, k, v, do, sel, vbs = _inputs(be, D, 1, 6, 6, 9)
    q[..., 3] = q[..., 3].abs() + 0.5
    clean = _run(q, k, v, do, sel, vbs, be)[0]
    # a key at -inf has weight zero
    k1, k2 = k.clone(), k.clone()
    k1[0, 0, 5, 3] = -math.inf
    k2[0, 0, 5, 3] = -1e30
    out1, out2 = (_run(q, x, v, do, sel, vbs, be)[0] for x in (k1, k2))
    assert torch.equal(out1, out2)
    # every query sees the key (topk = blocks): an infinite value fills its column
    v1 = v.clone()
    v1[0, 0, 5, 7] = math.inf
    out = _run(q, k, v1, do, sel, vbs, be)[0]
    assert (out[..., 7] == math.inf).all()
    rest = [d for d in range(D) if d != 7]
    assert torch.equal(out[..., rest], clean[..., rest])
    # the largest finite values stay finite (no weight is above 1)
    v1[0, 0, 5, 7] = torch.finfo(torch.float32).max
    out = _run(q, k, v1, do, sel, vbs, be)[0]
    assert torch.isfinite(out).all() and (out[..., 7] > 1e33).all()
    # a NaN query row is NaN and no other row is touched
    q1 = q.clone()
    q1[0, 0, 40, 2] = math.nan
    out = _run(q1, k, v, do, sel, vbs, be)[0]
    assert torch.isnan(out[0, 0, 40]).all()
    rows = [i for i in range(out.shape[2]) if i != 40]
    assert torch.equal(out[0, 0, rows], clean[0, 0, rows])
