"""The forward launched in pieces (block 64, key sequences past the L2 cache, long
routes) gives what one launch gives: the query blocks in one call against the
same blocks in calls too small to be split, around the sizes where a further
piece begins."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(autouse=True)
def _gpu_only():
    if not torch.cuda.is_available():
        pytest.skip("needs an MI355X")


def _attend(q, k, v, sel, vbs, be):
    from vsa_mi355x import mi355x as M
    return M.mi355x_sparse_attention(q, k, v, sel, vbs, block_size=(1, 1, be))


# query blocks in all beside a multiple of what the chip holds at once (per CU:
# four workgroups at head dim 128, eight at 64)
@pytest.mark.parametrize("d,per_cu,kb,tk,be", [(128, 4, 384, 48, 64), (64, 8, 1280, 160, 64),
                                               (128, 4, 400, 50, 33)])
@pytest.mark.parametrize("pieces,off", [(10, -1), (10, 0), (10, 1), (11, -3), (12, 5)])
def test_pieces_equal_single_launches(d, per_cu, kb, tk, be, pieces, off):
    H = 4
    resident = torch.cuda.get_device_properties(0).multi_processor_count * per_cu
    qb = pieces * resident // H + off
    g = torch.Generator(device=DEV).manual_seed(qb + d)
    q = torch.randn(1, H, qb * be, d, generator=g, device=DEV).bfloat16()
    k, v = (torch.randn(1, H, kb * be, d, generator=g, device=DEV).bfloat16() for _ in range(2))
    sel = torch.argsort(torch.rand(1, H, qb, kb, generator=g, device=DEV), -1)[..., :tk]
    sel = sel.sort(-1).values.int()
    vbs = torch.randint(1, be + 1, (kb,), generator=g, device=DEV, dtype=torch.int32)
    with torch.no_grad():
        got = _attend(q, k, v, sel, vbs, be)
        for i in range(0, qb, resident):
            n = min(resident, qb - i)
            ref = _attend(q[:, :, i * be:(i + n) * be].contiguous(), k, v,
                          sel[:, :, i:i + n].contiguous(), vbs, be)
            assert torch.equal(got[:, :, i * be:(i + n) * be], ref), i


def test_token_major_views_in_pieces():
    """The raster instance of the kernel: all heads in one call, which is split,
    against nine heads a call, which are not (10 368 and 3 456 workgroups)."""
    from vsa_mi355x import mi355x as M
    H, nb, tk, d = 27, 384, 48, 128
    g = torch.Generator(device=DEV).manual_seed(7)
    q, k, v = (torch.randn(1, nb * 64, H, d, generator=g, device=DEV).bfloat16() for _ in range(3))
    vbs = torch.randint(1, 65, (nb,), generator=g, device=DEV, dtype=torch.int32)

    def op(h):
        views = (x[:, :, h].contiguous().transpose(1, 2) for x in (q, k, v))
        return M.mi355x_vsa(*views, vbs, vbs, tk, (4, 4, 4))

    with torch.no_grad():
        got = op(slice(None))
        for i in range(0, H, 9):
            assert torch.equal(got[:, i:i + 9], op(slice(i, i + 9))), i
