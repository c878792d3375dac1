"""Errors of the fp32 kernels at head dims 64 / 128 (split bf16 products) that
random data does not show."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
SHAPES = [(64, 64), (64, 128), (128, 64), (256, 64), (256, 128)]


@pytest.fixture(autouse=True)
def _gpu_only():
    if not torch.cuda.is_available():
        pytest.skip("needs an MI355X")


def _own_block(H, nb):
    """Every query block routed to its own key block, of which one key is valid."""
    sel = torch.arange(nb, device=DEV, dtype=torch.int32).view(1, 1, nb, 1)
    return sel.expand(1, H, nb, 1).contiguous(), torch.ones(nb, dtype=torch.int32, device=DEV)


@pytest.mark.parametrize("be,D", SHAPES)
def test_infinite_gradients_stay_infinite(be, D):
    """One infinite value in dO makes its row of dS -inf at the keys whose v has
    the other sign there: those keys' dK is infinite with the sign of -q, the
    other keys' NaN."""
    from vsa_mi355x import mi355x as M
    nb = 3
    g = torch.Generator(device=DEV).manual_seed(be + D)
    q, k, v, do = (torch.randn(1, 1, be * nb, D, generator=g, device=DEV) for _ in range(4))
    sel = torch.arange(nb, device=DEV, dtype=torch.int32).expand(1, 1, nb, nb).contiguous()
    vbs = torch.full((nb,), be, dtype=torch.int32, device=DEV)
    do[0, 0, 40, 3] = math.inf
    leaves = [x.clone().requires_grad_() for x in (q, k, v)]
    out = M.mi355x_sparse_attention(*leaves, sel, vbs, block_size=(1, 1, be))
    got = torch.autograd.grad(out, leaves, do)[1][0, 0].double()
    q, k, v, do = (x[0, 0].double().cpu() for x in (q, k, v, do))
    p = torch.softmax(q @ k.T / math.sqrt(D), -1)
    delta = ((p @ v) * do).sum(-1, keepdim=True)
    ref = ((p * (do @ v.T - delta)).T @ q / math.sqrt(D)).to(DEV)
    assert torch.isinf(ref).any() and torch.isnan(ref).any()
    assert torch.equal(torch.isnan(got), torch.isnan(ref))
    assert torch.equal(got[torch.isinf(ref)], ref[torch.isinf(ref)])


@pytest.mark.parametrize("be,D", SHAPES)
def test_weights_come_from_the_scores_of_the_forward(be, D):
    """With one key a row and exponents of exactly the score (scale ln 2, whose
    product with log2 e rounds to 1), P is exp2(S - S): 1 exactly if dK / dV sums
    S as the forward does, so dV is what it is for scores of zero."""
    from vsa_mi355x import mi355x as M
    nb, H = 5, 3
    g = torch.Generator(device=DEV).manual_seed(be + D)
    q, k, v, do = (1 + torch.rand(1, H, be * nb, D, generator=g, device=DEV) for _ in range(4))
    sel, vbs = _own_block(H, nb)

    def dv(q):
        leaves = [x.clone().requires_grad_() for x in (q, k, v)]
        out = M.mi355x_sparse_attention(*leaves, sel, vbs, block_size=(1, 1, be),
                                        sm_scale=0.6931471824645996)
        return torch.autograd.grad(out, leaves, do)[2]

    assert torch.equal(dv(q), dv(torch.zeros_like(q)))


@pytest.mark.parametrize("be,D", SHAPES)
def test_lse_of_one_key_is_its_score(be, D):
    """Scores of whole numbers are exact: the log-sum-exp of a row of one key is
    its score times scale log2 e, rounded once."""
    from vsa_mi355x import mi355x as M
    nb, H, scale = 5, 3, 0.01
    g = torch.Generator(device=DEV).manual_seed(be + D)
    q, k = (torch.randint(-3, 4, (1, H, be * nb, D), generator=g, device=DEV).float()
            for _ in range(2))
    sel, vbs = _own_block(H, nb)
    lse = M.sparse_forward(q, k, k, sel, vbs, be, scale)[1].view(H, nb, be)
    keys = k.view(H, nb, be, 1, D)[:, :, :1, 0]
    s = (q.view(H, nb, be, D) * keys).sum(-1)
    c2 = torch.tensor(scale, dtype=torch.float32) * torch.tensor(math.log2(math.e))
    assert torch.equal(lse, s * c2.to(DEV))
