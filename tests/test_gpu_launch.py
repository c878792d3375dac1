"""A pass launched by one call gives, bit for bit, what the same steps give called
one by one (``return_aux=True`` runs them so): native, padded and token-major
shapes, every gate kind, each type, ragged blocks, unequal lengths, and the
fine branch on a route.  The block moves of padded shapes take 16-, 8-, 4- and
2-byte units."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF, HF, F = torch.bfloat16, torch.float16, torch.float32


@pytest.fixture(autouse=True)
def _gpu_only():
    if not torch.cuda.is_available():
        pytest.skip("needs an MI355X")


def _same(a, b, names):
    for n, x, y in zip(names, a, b):
        assert x.shape == y.shape and x.dtype == y.dtype and torch.equal(x, y), n


def _rand(seed, shapes, dt):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return [torch.randn(s, generator=g, device=DEV).to(dt) for s in shapes]


# (block volume, head dim, query blocks, key blocks, type, gate): unit of the moves in brackets
CASES = [(64, 64, 5, 5, BF, "full"), (256, 128, 3, 4, HF, "token"), (128, 256, 3, 3, BF, None),
         (64, 128, 4, 4, F, "full"), (64, 128, 4, 4, BF, "f32"), (128, 64, 3, 3, BF, "tokmaj"),
         (27, 80, 7, 9, BF, "full"),      # 16
         (100, 68, 3, 5, HF, "token"),    # 8, gate 2
         (64, 42, 6, 6, BF, "f32"),       # 4, gate 8
         (1, 33, 9, 7, BF, "full"),       # 2
         (127, 192, 3, 3, BF, "tokmaj"),  # 16
         (65, 30, 4, 4, F, "token"),      # 8, gate 4
         (3, 1, 5, 5, BF, "full")]        # 2


@pytest.mark.parametrize("be,d,qb,kb,dt,kind", CASES)
def test_full_op_equals_its_steps(be, d, qb, kb, dt, kind):
    from vsa_mi355x import mi355x as M
    B, H = 2, 3
    q, k, v, do = _rand(be + d, [(B, H, n * be, d) for n in (qb, kb, kb, qb)], dt)
    g = torch.Generator(device=DEV).manual_seed(1)
    gate = None
    if kind is not None:
        width = 1 if kind == "token" else d
        shape = (B, qb * be, H, width) if kind == "tokmaj" else (B, H, qb * be, width)
        gate = torch.rand(shape, generator=g, device=DEV, dtype=F if kind == "f32" else dt)
        gate = gate.transpose(1, 2) if kind == "tokmaj" else gate
    vbs, qvbs = (torch.tensor([max(1, be - 3 * i) for i in range(n)], dtype=torch.int32,
                              device=DEV) for n in (kb, qb))

    def step(aux):
        leaves = [x.detach().requires_grad_() for x in (q, k, v, gate) if x is not None]
        r = M.mi355x_vsa(*leaves[:3], vbs, qvbs, 2, (1, 1, be),
                         leaves[3] if gate is not None else None, return_aux=aux)
        out = r[0] if aux else r
        return [out.detach(), *torch.autograd.grad(out, leaves, do)]

    names = ["out", "dq", "dk", "dv", "dgate"]
    got, ref = step(False), step(True)
    _same(got, ref, names)
    with torch.no_grad():
        out = M.mi355x_vsa(q, k, v, vbs, qvbs, 2, (1, 1, be), gate)
    assert torch.equal(out, ref[0])


@pytest.mark.parametrize("be,d,dt", [(64, 64, BF), (256, 128, HF), (27, 80, BF), (100, 64, F)])
def test_route_op_equals_its_steps(be, d, dt):
    from vsa_mi355x import mi355x as M
    B, H, qb, kb, tk = 1, 3, 5, 8, 3
    q, k, v, do = _rand(be + d, [(B, H, n * be, d) for n in (qb, kb, kb, qb)], dt)
    sel = torch.argsort(torch.rand(B, H, qb, kb, device=DEV), -1)[..., :tk].int()
    vbs = torch.tensor([max(1, be - 2 * i) for i in range(kb)], dtype=torch.int32, device=DEV)
    leaves = [x.requires_grad_() for x in (q, k, v)]
    out = M.mi355x_sparse_attention(*leaves, sel, vbs, block_size=(1, 1, be), sm_scale=0.2)
    got = [out.detach(), *torch.autograd.grad(out, leaves, do)]
    # the steps on torch-padded tensors
    kbe, kd = M._kernel_block(be), M._kernel_dim(d)

    def pad(x):
        x = x.detach().view(B, H, -1, be, d)
        return torch.nn.functional.pad(x, (0, kd - d, 0, kbe - be)).reshape(B, H, -1, kd)

    def unpad(x):
        return x.view(B, H, -1, kbe, kd)[..., :be, :d].reshape(B, H, -1, d)

    qp, kp, vp, dp = (pad(x) for x in (q, k, v, do))
    o, lse, _ = M.sparse_forward(qp, kp, vp, sel, vbs, kbe, 0.2)
    delta, _, _ = M.backward_prep(o, dp, kbe)
    grads = M.sparse_backward(qp, kp, vp, dp, lse, delta, sel, vbs, kbe, 0.2)
    _same(got, [unpad(x) for x in (o, *grads)], ["out", "dq", "dk", "dv"])


def test_saved_tensors_come_back_unaligned():
    """A saved-tensor hook may give the kept workspace back at any address."""
    from vsa_mi355x import mi355x as M
    q, k, v, do = (x.requires_grad_() for x in _rand(3, [(1, 2, 320, 64)] * 4, BF))
    vbs = torch.full((5,), 64, dtype=torch.int32, device=DEV)

    def unpack(t):
        if t.dtype != torch.uint8:
            return t
        return torch.empty(t.numel() + 16, dtype=torch.uint8, device=DEV)[16:].copy_(t)

    def grads():
        return torch.autograd.grad(M.mi355x_vsa(q, k, v, vbs, vbs, 2, (4, 4, 4)), [q, k, v],
                                   do.detach())

    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
        got = grads()
    _same(got, grads(), ["dq", "dk", "dv"])
