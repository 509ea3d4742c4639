"""Fused window attention: token plans and the call into the compiled host path (``csrc/native.cpp``), which runs the
attention, or the attention with the two dense layers around it, as one autograd node.

Numerically this is the same computation as the operator-by-operator composition in
:mod:`sparseswin3d_amd.window_attention` (reference ``sparse_swin/swin3d_base.py:654-675``):

    S = (scale*Q) K^T + bias + mask  ->  P = sparse softmax(S)  ->  O = P V  (in voxel order)

but Q, K, V token rows are read straight from the dense ``qkv`` tensor through the token order
and the output is written straight into voxel order, so the sorted COO copies, the bias/mask
gather passes, the permute and the un-sort never exist.  Three families of kernels (:func:`attention_path`): two keep the
attention matrix in registers and form it again in the backward pass, the block products keep P in memory.
"""
from __future__ import annotations

import ctypes as C

import torch

from . import _lib

_DTYPE_CODE = {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}


def _ptr(t):
    return C.c_void_p(t.data_ptr() if t is not None else 0)


class TokenPlan:
    """Token order and per-group table of one set of (window, pos) voxel indices.

    With ``defer=True`` the constructor only enqueues the kernels, the last of which writes the totals to pinned memory;
    work enqueued afterwards (the qkv projection) overlaps the host round trip, and
    :meth:`finish` waits for the totals when they are needed.  :meth:`finish` raises if an index
    lies outside ``[0, batch_size) x [0, n)`` or a (window, pos) pair occurs twice, and so does every later use of the plan.

    ``tokens``, ``plan`` and ``tasks`` are the device tables of ``sswin_token_plan``; ``tasks``: group descriptors of the
    window-resident kernels, bucketed by ceil(c / 32), and behind them the token records, one per window and tile of 32
    tokens.  ``order_only``: the plan of a stride-2 merge, whose consumers read the voxel of every rank and nothing else."""

    def __init__(self, indices: torch.Tensor, batch_size: int, n: int, num_heads: int, defer: bool = False,
                 tasks: bool = True, order_only: bool = False):
        self._allocate(indices, batch_size, n, num_heads, tasks, order_only)
        _lib.native().enqueue_plans([self.native])
        if not defer:
            self.finish()

    def _allocate(self, indices, batch_size, n, num_heads, tasks, order_only=False):
        self.native = _lib.native().Plan(indices, int(batch_size), int(n), int(num_heads), tasks, order_only)

    @classmethod
    def batch(cls, specs):
        """Deferred plans for several index sets on one device, built by shared launches (the regular and the
        shifted block of a stage).  ``specs``: tuples ``(indices, batch_size, n, num_heads)``,
        ``(..., tasks)`` or ``(..., tasks, order_only)``; returns the plans in the same order, each to be completed
        with :meth:`finish`."""
        plans = []
        for spec in specs:
            p = cls.__new__(cls)
            p._allocate(*spec[:4], spec[4] if len(spec) > 4 else True, spec[5] if len(spec) > 5 else False)
            plans.append(p)
        if plans:
            _lib.native().enqueue_plans([p.native for p in plans])
        return plans

    def finish(self):
        """Wait for the totals (once) and decode them."""
        self.native._finish()
        return self

    @property
    def bucket_counts(self):
        """Groups per number of 32-token tiles (1..4), as the library's entry points take them."""
        return (C.c_int64 * 4)(*self.native.buckets)


for _name in ("tokens", "plan", "tasks", "device", "N", "H", "n", "B", "g_cap", "order_only", "G", "windows", "A", "c_max",
              "oversize_groups"):
    setattr(TokenPlan, _name, property(lambda self, _name=_name: getattr(self.native, _name)))


def _group_softmax(tp, backward, x_or_y, grad, out):
    """Row softmax (or its backward) over the [c x c] blocks of the plan's groups; ``out`` may be one of the inputs."""
    _lib.check(_lib.load().sswin_group_softmax(
        1 if backward else 0, _ptr(tp.plan), tp.g_cap, tp.G, tp.N, tp.H, tp.c_max, _ptr(x_or_y), _ptr(grad), _ptr(out),
        _lib.stream_handle(tp.device)))


def _bias_gradient(tp, d_s, bias_meta, table_index):
    """Gradient of the [H, n, n] bias, or of the [rows, H] table when ``table_index`` is given, from dS
    (one [c x c] block per group)."""
    dtype, shape = bias_meta
    code, offset0 = (None, 0) if table_index is None else (table_index.code, table_index.offset0)
    return _lib.native().bias_gradient(tp.native, d_s, code, offset0, list(shape), dtype)


class BiasTableIndex:
    """The relative position index [n, n] of a bias table in the form the library uses:
    ``index[p, q] = code[p] - code[q] + offset0`` (true for the index arithmetic of
    sparse_swin/swin3d_base.py:630-647).  :meth:`build` returns None if an index is not of
    that form or the table is too large for the table-gradient kernel."""

    def __init__(self, flat, code, offset0, ascending=False):
        self.flat, self.code, self.offset0 = flat, code, offset0
        self.ascending = ascending          # no negative code: what the kernels that read the table itself take

    @staticmethod
    def build(index: torch.Tensor, table_rows: int):
        n = index.shape[0]
        if index.dim() != 2 or index.shape[1] != n or n > 384 or table_rows > 4096 or n == 0:
            return None
        idx = index.to(torch.int64)
        # index[p, q] = code[p] - code[q] + offset0 with code[0] = 0; every check in one read from the device
        code = idx[:, 0] - idx[0, 0]
        linear, low, high, offset0, first = torch.stack([
            (idx == code[:, None] - code[None, :] + idx[0, 0]).all().to(torch.int64), idx.min(), idx.max(), idx[0, 0], code.min()]).tolist()
        if not linear or low < 0 or high >= table_rows:
            return None
        return BiasTableIndex(idx.reshape(-1).contiguous(), code.to(torch.int32).contiguous(), offset0, first >= 0)


def fused_window_attention(qkv, bias, indices, mask, batch_size, n, scale, resident=None, plan=None,
                           table_index=None, projections=None):
    """``qkv`` [N,3,H,hd], ``bias`` [H,n,n], ``indices`` int32 [N,2] (window,pos), ``mask`` int8
    [nW,n] or None -> attention output [N, H*hd] in the caller's voxel order.

    ``resident``: None = the kernels that keep the attention matrix in registers wherever they apply (:func:`attention_path`),
    True = the window-resident ones (heads of 32 channels), False = block products with the attention matrix in HBM.
    ``plan``: a :class:`TokenPlan` of ``indices`` made earlier (possibly still in flight).
    ``table_index``: a :class:`BiasTableIndex`; ``bias`` is then the [rows, H] bias table and its
    gradient is computed without the [H, n, n] detour.
    ``projections``: (features [N, D], qkv layer, proj layer, heads, compute dtype) in place of ``qkv``: the two dense
    layers around the attention run in the same autograd node and the result is the projected output."""
    code, offset0 = (None, 0) if table_index is None else (table_index.code, table_index.offset0)
    if projections is not None:
        features, to_qkv, proj, heads, dtype = projections
        tp = plan if plan is not None else TokenPlan(indices, batch_size, n, heads, defer=True)
        return _lib.native().attention_module(features, to_qkv.weight, to_qkv.bias, bias, proj.weight, proj.bias, tp.native, mask, code,
                                              offset0, n, heads, scale,
                                              attention_path(features.shape[1] // heads, n, table_index, resident), dtype)
    tp = plan if plan is not None else TokenPlan(indices, batch_size, n, qkv.shape[2], defer=True)
    return _lib.native().attention(qkv, bias, tp.native, mask, code, offset0, int(n), float(scale),
                                   attention_path(qkv.shape[3], n, table_index, resident))


def attention_path(head_dim: int, n: int, table_index, resident=None) -> str:
    """Which kernels run an attention the fused path takes.  "resident": heads of 32 channels, windows of at most 128 positions;
    "flash": heads of 16 or 32 channels and any window, the bias read from the relative position table; "products": block
    products with the attention matrix in memory (any head size)."""
    if resident or (resident is None and head_dim == 32 and n <= 128):
        return "resident"
    if resident is None and head_dim in (16, 32) and table_index is not None and table_index.ascending:
        return "flash"
    return "products"


def supports(qkv: torch.Tensor, n: int, table: bool = False) -> bool:
    """The fused path covers fp32/fp16/bf16 on the GPU.  Windows: at most 128 positions when the bias gradient is
    formed as an [H, n, n] array (its LDS table), at most 384 (7^3 = 343 included) when it goes straight to the
    relative position table (``table``: the module has a :class:`BiasTableIndex`).  Everything else takes the
    operator-by-operator path."""
    return qkv.is_cuda and qkv.dtype in _DTYPE_CODE and (n <= 384 if table else n * n * 4 <= 64 * 1024)
