"""The one-call passes' sizes and argument checks (no GPU needed)."""

import ctypes

from vsa_mi355x import _lib, launch


def _spec(**kw):
    base = dict(bh=2, sq=256, skv=512, s_out=0, heads=0, head_dim=64, block=64, kernel_dim=64,
                kernel_block=64, topk=2, gate_mode=0, gate_heads=1, dtype=0, keep=1, scale=0.1,
                route=False)
    return launch.Spec(**{**base, **kw})


def test_sizes_follow_the_op():
    full, route = launch._sizes(_spec()), launch._sizes(_spec(route=True))
    # kept: pooled rows, probabilities, route, fine output, lse; the route op keeps the lse alone
    assert full[0] > route[0] == 2 * 256 * 4
    assert launch._sizes(_spec(keep=0))[0] == 0
    padded = launch._sizes(_spec(block=32))   # twice the rows, and copies of q, k, v
    assert padded[0] > 2 * full[0]
    assert launch._sizes(_spec(s_out=250, skv=256))[0] > full[0]
    assert all(x % 256 == 0 for x in (*full, *route, *padded))


def _rc(fn, spec, *args, rows=None, selected=None):
    op = launch._struct(spec, 256, 256, 256, None, selected, 256, 256, rows)
    return getattr(_lib.load(), fn)(ctypes.byref(op), *args)


def test_bad_arguments_are_refused_before_any_launch():
    n = (ctypes.c_int64 * 3)()
    at = [ctypes.addressof(n) + 8 * i for i in range(3)]
    assert _lib.load().vsa_op_sizes(None, *at) == -1
    assert _rc("vsa_op_sizes", _spec(), at[0], None, at[2]) == -1
    assert _rc("vsa_op_sizes", _spec(dtype=7), *at) == -3
    assert _rc("vsa_op_sizes", _spec(sq=250), *at) == -2              # not whole blocks
    assert _rc("vsa_op_sizes", _spec(head_dim=65), *at) == -2         # wider than its kernel
    assert _rc("vsa_op_sizes", _spec(topk=0), *at) == -2
    assert _rc("vsa_op_sizes", _spec(block=32), *at, rows=256) == -2  # raster tokens, padded
    assert _rc("vsa_op_sizes", _spec(), *at, rows=256, selected=256) == -2
    assert _rc("vsa_op_fwd", _spec(), None, 256, 256, None) == -1     # no out
    assert _rc("vsa_op_fwd", _spec(), 256, None, 256, None) == -1     # nothing to keep into
    assert _rc("vsa_op_fwd", _spec(), 256, 256, None, None) == -1     # no scratch
    assert _rc("vsa_op_fwd", _spec(), 256, 264, 256, None) == -7
    assert _rc("vsa_op_fwd", _spec(gate_mode=1), 256, 256, 256, None) == -1   # no gate
    assert _rc("vsa_op_bwd", _spec(), None, 256, 256, 256, 256, 256, None, None, None) == -1
    assert _rc("vsa_op_bwd", _spec(keep=0), None, 256, 256, 256, 256, 256, 256, None, None) == -1
