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


def _dp(be, v, do):
    """dP of each row of dO with its block's first row of v: dQ with P = 1 (scores
    and log-sum-exp of zero), delta = 0, and a key of ones."""
    from vsa_mi355x import mi355x as M
    _, H, S, D = do.shape
    sel, vbs = _own_block(H, S // be)
    zero = torch.zeros(1, H, S, device=DEV)
    dq = M.sparse_backward(torch.zeros_like(do), torch.ones_like(do), v, do, zero, zero, sel, vbs,
                           be, 1.0)[0]
    assert torch.equal(dq[..., :1].expand_as(dq), dq)
    first = v.view(H, S // be, be, D)[:, :, :1].expand(H, S // be, be, D).double()
    return dq[..., 0].double(), (first * do.view(H, S // be, be, D).double()).sum(-1).view(1, H, S)


@pytest.mark.parametrize("be,D", SHAPES)
@pytest.mark.parametrize("size", [1.0, 1e-35, 1e-37])
def test_single_products(be, D, size):
    """What the six partial products leave out is at most 2^-24 of a product (its
    mid and lo parts are at most 2^-8 and 2^-17 of the leading bits: 2 * 2^-25),
    the sum's rounding 2^-24, and the sum of what is smaller well under a quarter
    of that.  Parts below 2^-133 do not exist: as much is lost of each factor and
    of dS."""
    g = torch.Generator(device=DEV).manual_seed(be + D)
    nb, H = 8, 4
    worst = torch.tensor([1 + 2.0 ** -7 - 2.0 ** -23, 1 + 2.0 ** -8, 1 + 2.0 ** -8 - 2.0 ** -17,
                          1 + 2.0 ** -8 + 2.0 ** -16 - 2.0 ** -23, 2 - 2.0 ** -23], device=DEV)
    v, do = (torch.zeros(1, H, be * nb, D, device=DEV) for _ in range(2))
    for x in (v, do):
        x[..., 5] = 1 + torch.rand(x.shape[:3], generator=g, device=DEV)
        pick = torch.randint(0, 10, x.shape[:3], generator=g, device=DEV)
        x[..., 5] = torch.where(pick < 5, worst[pick.clamp(max=4)], x[..., 5])
    got, ref = _dp(be, v, do * size)
    err = (got - ref).abs() / (2.25 * 2.0 ** -24 * ref.abs() + 4 * 2.0 ** -133)
    print(f"  be={be} D={D}: {err.max().item():.3f} of the bound", flush=True)
    assert err.max() <= 1


@pytest.mark.parametrize("be,D", SHAPES)
def test_same_signed_products(be, D):
    """Operands of one sign and nearly one value: the error is that of 6 D / 16
    independent roundings of the sum (2^-24 / sqrt 3 each), with no common part."""
    g = torch.Generator(device=DEV).manual_seed(be + D)
    v, do = (1 + 2.0 ** -7 - 2.0 ** -23 * torch.randint(0, 16, (1, 4, be * 8, D), generator=g,
                                                        device=DEV) for _ in range(2))
    got, ref = _dp(be, v, do)
    rms = ((got - ref) / ref).pow(2).mean().sqrt().item()
    print(f"  be={be} D={D}: {rms:.2e}", flush=True)
    assert rms <= math.sqrt(6 * D / 16 / 3) * 2.0 ** -24
