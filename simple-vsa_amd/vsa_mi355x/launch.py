"""A whole pass of an op as one call into the C ABI (``vsa_op_fwd`` /
``vsa_op_bwd``), and the autograd Function around the two.

The host side of a small pass costs more than its kernels: each separate call
from Python converts its arguments, allocates its outputs and looks up the
stream.  Here a pass is one struct, one workspace the backward needs
(``saved``), one it does not (``scratch``) and one call; the layout of the
workspaces is the library's own.  Covers the full op, the fine branch on a
caller's route, raster-order tokens, and shapes zero-padded onto the kernels
(triton_impl.py:1530-1580, 1655-1731).
"""

from __future__ import annotations

import contextlib
import ctypes
import functools
from typing import NamedTuple, Optional

import torch
from torch import Tensor
from torch.autograd.function import once_differentiable

from . import _lib

_NO_CONTEXT = contextlib.nullcontext()


def on_device(device: torch.device):
    """``torch.cuda.device(device)``, free when it is the current one already."""
    if torch._C._cuda_getDevice() == device.index:
        return _NO_CONTEXT
    return torch.cuda.device(device)


class Spec(NamedTuple):
    """The sizes and options of an op: plain values, so that equal specs share a plan."""
    bh: int
    sq: int          # the caller's lengths; nb * block for raster tokens
    skv: int
    s_out: int       # raster tokens per head, 0 otherwise
    heads: int       # heads of token-major raster tokens, 0 otherwise
    head_dim: int
    block: int
    kernel_dim: int
    kernel_block: int
    topk: int
    gate_mode: int
    gate_heads: int
    dtype: int
    keep: int
    scale: float
    route: bool      # the caller's route instead of the coarse branch

    @property
    def copies(self) -> bool:
        """The forward keeps its own copies of q, k and v."""
        return self.s_out > 0 or self.padded

    @property
    def padded(self) -> bool:
        return self.kernel_dim != self.head_dim or self.kernel_block != self.block


def _struct(spec: Spec, q, k, v, gate, selected, vbs, qvbs, rows) -> _lib.VsaOp:
    return _lib.VsaOp(q, k, v, gate, selected, vbs, qvbs, rows, *spec[:15])


@functools.lru_cache(maxsize=256)
def _sizes(spec: Spec):
    """Bytes of (saved, forward scratch, backward scratch)."""
    some = 256  # any non-null pointer: only its presence is read
    op = _struct(spec, None, None, None, None, some if spec.route else None, None, None,
                 some if spec.s_out else None)
    n = (ctypes.c_int64 * 3)()
    at = ctypes.addressof(n)
    _lib.call("vsa_op_sizes", ctypes.byref(op), at, at + 8, at + 16)
    return tuple(n)


def _ptr(t: Optional[Tensor]):
    return None if t is None else t.data_ptr()


def _workspace(n: int, device: torch.device) -> Optional[Tensor]:
    return torch.empty(n, dtype=torch.uint8, device=device) if n else None


def forward(spec: Spec, q, k, v, gate, selected, vbs, qvbs, rows, out):
    """Run the forward into ``out``; returns ``saved`` (None with nothing kept)."""
    dev = q.device
    n_saved, n_scratch, _ = _sizes(spec)
    saved, scratch = _workspace(n_saved, dev), _workspace(n_scratch, dev)
    op = _struct(spec, q.data_ptr(), k.data_ptr(), v.data_ptr(), _ptr(gate), _ptr(selected),
                 vbs.data_ptr(), _ptr(qvbs), _ptr(rows))
    _lib.call("vsa_op_fwd", ctypes.byref(op), out.data_ptr(), _ptr(saved), _ptr(scratch),
              torch._C._cuda_getCurrentRawStream(dev.index))
    return saved


class Op(torch.autograd.Function):
    """The op as a differentiable function of q, k, v and the gate."""

    @staticmethod
    def forward(ctx, spec, q, k, v, gate, selected, vbs, qvbs, rows):
        out = torch.empty_like(q)
        saved = forward(spec, q, k, v, gate, selected, vbs, qvbs, rows, out)
        ctx.spec = spec
        ctx.like = (q.shape, k.shape, gate.shape if gate is not None else None,
                    gate.dtype if gate is not None else None)
        ctx.save_for_backward(
            *((None,) * 3 if spec.copies else (q, k, v)), None if spec.padded else gate, selected,
            vbs, qvbs, rows, out if spec.route and not spec.padded else None, saved)
        return out

    @staticmethod
    @once_differentiable
    def backward(ctx, dout):
        spec = ctx.spec
        q, k, v, gate, selected, vbs, qvbs, rows, out, saved = ctx.saved_tensors
        q_shape, k_shape, gate_shape, gate_dtype = ctx.like
        dout = dout.contiguous()
        if dout.data_ptr() % 16:
            dout = dout.clone()
        if saved.data_ptr() % 256:  # what a saved-tensor hook gave back
            saved = saved.clone()
        dev = dout.device
        dq = torch.empty(q_shape, dtype=dout.dtype, device=dev)
        dk = torch.empty(k_shape, dtype=dout.dtype, device=dev)
        dv = torch.empty_like(dk)
        d_gate = None
        if gate_shape is not None:
            if (spec.gate_mode & ~_lib.GATE_F32) == _lib.GATE_TOKEN_MAJOR:
                b, h, s, d = gate_shape   # the gate's own layout
                d_gate = torch.empty((b, s, h, d), dtype=gate_dtype, device=dev).transpose(1, 2)
            else:
                d_gate = torch.empty(gate_shape, dtype=gate_dtype, device=dev)
        scratch = _workspace(_sizes(spec)[2], dev)
        op = _struct(spec, _ptr(q), _ptr(k), _ptr(v), _ptr(gate), _ptr(selected), vbs.data_ptr(),
                     _ptr(qvbs), _ptr(rows))
        _lib.call("vsa_op_bwd", ctypes.byref(op), _ptr(out), dout.data_ptr(), saved.data_ptr(),
                  _ptr(scratch), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), _ptr(d_gate),
                  torch._C._cuda_getCurrentRawStream(dev.index))
        return None, dq, dk, dv, d_gate, None, None, None, None


def run(spec: Spec, q, k, v, gate, selected, vbs, qvbs, rows) -> Tensor:
    """The op on prepared tensors (contiguous, 16-byte aligned, on one device):
    through autograd where a gradient is wanted, else the forward alone.
    ``spec.keep`` is set here."""
    needs_grad = torch.is_grad_enabled() and (
        q.requires_grad or k.requires_grad or v.requires_grad
        or (gate is not None and gate.requires_grad))
    with on_device(q.device):
        if needs_grad:
            return Op.apply(spec._replace(keep=1), q, k, v, gate, selected, vbs, qvbs, rows)
        out = torch.empty_like(q)
        forward(spec, q, k, v, gate, selected, vbs, qvbs, rows, out)
        return out
