"""The coarse kernels at the sizes where they change path: key tiles per wave kept
in registers (up to 256, 512 and 768 blocks), tiles shared by one or two waves
per partial sum (128 blocks), head dim 256 in two halves; the Top-K at its
register counts (64, 128, .. 2048 keys) on ties that do and do not resolve in
the upper half of the key; the CSR scan past its unrolled strides."""

import numpy as np
import pytest
import torch

from oracle import vsa_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(autouse=True)
def _gpu_only():
    if not torch.cuda.is_available():
        pytest.skip("needs an MI355X")


@pytest.mark.parametrize("D,qb,kb", [(64, 40, 128), (64, 33, 129), (128, 9, 256), (128, 31, 257),
                                     (64, 20, 513), (128, 129, 768), (64, 257, 769),
                                     (256, 5, 3), (256, 33, 130), (256, 70, 520), (256, 20, 769)])
def test_coarse_against_the_oracle(D, qb, kb):
    from vsa_mi355x import mi355x as M
    g = torch.Generator().manual_seed(D + qb + kb)
    qc, kc, vc, do = (torch.randn(1, 2, n, D, generator=g).bfloat16() for n in (qb, kb, kb, qb))
    scale = D ** -0.5
    dev = [x.to(DEV) for x in (qc, kc, vc)]
    _, probs, outc, _ = M.coarse_forward(*dev, None, scale)
    grads = M.coarse_backward(*dev, probs, do.to(DEV), scale)
    leaves = [t.clone().requires_grad_() for t in (qc, kc, vc)]
    ones_q, ones_k = torch.ones(qb, dtype=torch.long), torch.ones(kb, dtype=torch.long)
    _, out = O.coarse_branch_compact(*leaves, ones_k, ones_q, 1, scale)
    ref = torch.autograd.grad(out, leaves, do)
    # both round to bf16 (2^-9 relative) at the scores, the weights and the result
    for what, a, e in zip(("out_c", "d_q_c", "d_k_c", "d_v_c"), (outc, *grads), (out, *ref)):
        a, e = a.float().cpu(), e.detach().float()
        rel = ((a - e).norm() / e.norm()).item()
        assert rel <= 1e-2, (what, rel)


def test_columns_past_2_32_weights():
    """d_k_c and d_v_c of a head with more than 2^32 probabilities (16 000 key
    blocks; the last query rows lie past them): rows without weight add exact
    zeros and each key has one row with weight, so the rows that have some give
    the same by themselves, bit for bit."""
    from vsa_mi355x import mi355x as M
    kb, D = 16000, 64
    qb = (1 << 32) // kb + 100
    if torch.cuda.mem_get_info()[0] < 48 << 30:
        pytest.skip("needs 35 GB of free HBM")
    g = torch.Generator(device=DEV).manual_seed(1)
    qc, kc, vc, do = (torch.randn(1, 1, n, D, generator=g, device=DEV).bfloat16()
                      for n in (qb, kb, kb, qb))
    rows = torch.cat([torch.arange(40), torch.arange(qb - 150, qb)]).to(DEV)
    keys = torch.arange(rows.numel(), device=DEV) * 2
    probs = torch.zeros(1, 1, qb, kb, device=DEV)
    probs[0, 0, rows, keys] = 0.25
    probs[0, 0, rows, keys + 1] = 0.75
    got = M.coarse_backward(qc, kc, vc, probs, do, 0.125)
    ref = M.coarse_backward(qc[:, :, rows], kc, vc, probs[:, :, rows], do[:, :, rows], 0.125)
    assert all((x != 0).any() for x in ref)
    assert torch.equal(got[0][:, :, rows], ref[0])
    assert torch.equal(got[1], ref[1]) and torch.equal(got[2], ref[2])


@pytest.mark.parametrize("kb", [63, 64, 65, 128, 129, 512, 513, 1024, 1025, 2048, 2049])
@pytest.mark.parametrize("kind", ["bf16", "fp32", "low_bits", "few"])
def test_topk_against_the_rule(kb, kind):
    from vsa_mi355x import mi355x as M
    g = torch.Generator().manual_seed(kb)
    x = torch.randn(7, kb, generator=g)
    if kind == "bf16":       # ties that agree in the lower half of the key
        x = x.bfloat16().float()
    elif kind == "low_bits":  # ties of the upper half that differ in the lower
        x = (1.0 + torch.randint(0, 9, (7, kb), generator=g) * 2.0 ** -22) * \
            torch.where(torch.rand(7, kb, generator=g) < 0.5, 1.0, -1.0)
    elif kind == "few":       # one value but for a few
        x = torch.where(torch.rand(7, kb, generator=g) < 0.1, x, torch.tensor(-0.25))
    x[0, ::3] = -float("inf")
    for tk in sorted({1, 3, kb // 8, kb // 2, kb - 1, kb}):
        got = M.topk(x.to(DEV), tk).cpu().numpy()
        assert np.array_equal(got, np.sort(O.topk_reference(x, tk), axis=-1)), (kb, tk)


@pytest.mark.parametrize("qb,kb,tk", [(1, 3, 1), (64, 64, 8), (513, 40, 8), (60, 700, 513),
                                      (300, 300, 27)])
def test_csr_against_brute_force(qb, kb, tk):
    from vsa_mi355x import mi355x as M
    g = torch.Generator().manual_seed(qb + kb)
    sel = torch.argsort(torch.rand(1, 3, qb, kb, generator=g), -1)[..., :tk].int()
    sel[0, 1, qb // 2, 0] = -1
    sel[0, 2, qb // 3, tk - 1] = kb
    inv, off, cnt = (x.cpu() for x in M.invert_routes(sel.to(DEV), kb))
    for h in range(3):
        at = 0
        for k in range(kb):
            rows = (sel[0, h] == k).any(-1).nonzero().flatten().int()
            assert cnt[0, h, k] == len(rows) and off[0, h, k] == at
            assert torch.equal(inv[0, h, at:at + len(rows)], rows)
            at += len(rows)
