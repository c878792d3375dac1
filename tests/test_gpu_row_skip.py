"""Query rows that pad a block's volume take no products: volumes around the
32-row waves and the kernels' blocks, bit for bit what the steps give called one
by one, which multiply every row."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(autouse=True)
def _gpu_only():
    if not torch.cuda.is_available():
        pytest.skip("needs an MI355X")


def _same(a, b):
    for n, x, y in zip(["out", "dq", "dk", "dv", "dgate"], a, b):
        assert x.shape == y.shape and x.dtype == y.dtype and torch.equal(x, y), n


@pytest.mark.parametrize("d", [64, 96, 256])
@pytest.mark.parametrize("be", [2, 31, 32, 33, 63, 65, 96, 97, 127])
def test_padded_volume(be, d):
    from vsa_mi355x import mi355x as M
    B, H, n = 1, 2, 5
    g = torch.Generator(device=DEV).manual_seed(be + d)
    q, k, v, do = (torch.randn(B, H, n * be, d, generator=g, device=DEV).bfloat16()
                   for _ in range(4))
    gate = torch.rand(B, H, n * be, d, generator=g, device=DEV).bfloat16()
    vbs = torch.tensor([be, max(1, be - 1), be, 1, be], dtype=torch.int32, device=DEV)

    def step(aux):
        leaves = [x.detach().requires_grad_() for x in (q, k, v, gate)]
        r = M.mi355x_vsa(*leaves[:3], vbs, vbs, 2, (1, 1, be), leaves[3], return_aux=aux)
        out = r[0] if aux else r
        return [out.detach(), *torch.autograd.grad(out, leaves, do)]

    _same(step(False), step(True))
