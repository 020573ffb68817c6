"""``CUDABlockAttention``: sparse attention on a block mask, no key mask.

Drop-in for the reference module of the same name (models/attention_blockcuda.py): same constructor
``(config, attn_cpp, attn_handle)``, same ``forward(query, key, value, mask, mat)`` returning
``(out [B,H,L,d], P_flat [B*H*nnz])`` and the same autograd contract (gradients for query, key and value
only; the gradient of the returned probabilities is ignored, models/attention_blockcuda.py:73-112).
``attn_cpp`` is the ctypes library exporting init / attn_forward / attn_backward
(models/block_attn.cu:547-568), ``attn_handle`` the pointer its ``init`` returned.
"""
from __future__ import annotations

import ctypes

import torch
import torch.nn as nn

from . import _lib
from .csr import CsrCache


class _BlockAttnFunction(torch.autograd.Function):
    """The reference's function (models/attention_blockcuda.py:20-112) makes a transposed copy of K for the forward
    and of V for the backward because its ABI takes them that way, and its backward is not handed the forward's
    output.  Here every tensor stays row-major and autograd's saved ``out`` goes to the backward: the library's
    row-major calls (spion_attn_forward_scratch / spion_attn_backward_scratch) take them as they are.
    ``attn_cpp`` (the drop-in with the reference's four symbols) is still what created the handle.

    The reference also starts with ``.contiguous()`` copies of query, key and value (models/attention_blockcuda.py:
    36-48), which arrive as [B,H,L,d] views of [B,L,H*d] projections (models/attention.py:136-139).  The strided
    entry points read the views in place, write ``out`` in the same interleaved layout (so that combine_heads,
    models/attention.py:131-134, is a view as well) and the gradients likewise: no copy on either side of the
    kernels.  (Head dimension 64 on tile patterns is served the same way; its kernels read row-major K and V a cache
    line per lane, slower than the transposed form the contiguous entry points use, but still cheaper than the
    copies.)"""

    @staticmethod
    def forward(ctx, query, key, value, mask, mat, module):
        m = module
        shape = m.head_shape
        _lib.check_heads(shape, query, key, value, torch.float32)
        _lib.use_current_stream(m, query.device)
        idx = m.csr_cache.get(mat, m.block_size)
        nb_ = m.num_batches
        dev = query.device
        p_flat = torch.empty(nb_ * idx.nnz, dtype=torch.float32, device=dev)
        pen_ptr = None
        if m.with_mask:
            pen = (1e6 * (1.0 - mask.repeat(1, m.num_heads))).to(torch.float32).contiguous()  # [B, H*L]
            _lib.check_penalties(pen, shape, dev)
            pen_ptr = pen.data_ptr()
        lay = None
        if m.reads_views and not (query.is_contiguous() and key.is_contiguous() and value.is_contiguous()):
            lay = _lib.head_layout(query)
            if lay is None or key.stride() != query.stride() or value.stride() != query.stride() \
                    or _lib.head_layout(key) is None or _lib.head_layout(value) is None:
                lay = None
        if lay is not None:
            q, k, v = query, key, value
            out = _empty_heads(shape, interleaved=query.stride(1) < query.stride(2), device=dev)
        else:
            q, k, v = query.contiguous(), key.contiguous(), value.contiguous()
            out = torch.empty(shape, dtype=torch.float32, device=dev)
        lout = _lib.head_layout(out) if lay is not None else None
        scratch = _scratch(m, idx, False, dev)
        _lib.core().spion_attn_forward_scratch(
            m.attn_handle, q.data_ptr(), k.data_ptr(), v.data_ptr(), pen_ptr, 0, p_flat.data_ptr(), out.data_ptr(),
            *idx.tail[:2], idx.nnz, m.num_heads, _address(lay), _address(lout), *scratch[1:])
        _lib.check_error("attn_forward")
        _lib.save_for_backward(ctx, q, k, v, p_flat, out)
        ctx.set_materialize_grads(False)  # the gradient of the returned probabilities is ignored anyway
        ctx.module = m
        ctx.index = idx  # not among the saved tensors: the library knows it by its address
        ctx.strided = lay is not None
        if m.with_mask:
            ctx.mark_non_differentiable(p_flat)
        return out, p_flat

    @staticmethod
    def backward(ctx, grad_output, grad_weight):
        m = ctx.module
        q, k, v, p_flat, out = _lib.saved_tensors(ctx)
        p_flat, dev = p_flat.contiguous(), q.device
        _lib.use_current_stream(m, dev)
        if grad_output is None:  # only the probabilities were used downstream: their gradient is ignored
            grad_output = torch.zeros(m.batch_size, m.num_heads, m.seq_len, m.emb_dim, dtype=torch.float32, device=dev)
        lin = lout = lgrad = None
        if ctx.strided:
            (q, k, v), (out,) = _lib.one_layout(q, k, v), _lib.one_layout(out)
            go = grad_output
            if go.stride() != out.stride() or _lib.head_layout(go) is None:
                go = torch.empty_like(out).copy_(grad_output)  # preserves out's strides
            interleaved = q.stride(1) < q.stride(2)
            shape = tuple(q.shape)
            if _lib.adjacent_head_views(q, k, v):  # slices of one fused projection: the gradients likewise
                dq, dk, dv = _lib.empty_adjacent_heads(*shape, dev)
            else:
                dq, dk, dv = (_empty_heads(shape, interleaved, dev) for _ in range(3))
            lin, lout, lgrad = _lib.taken_layout(q), _lib.taken_layout(out), _lib.head_layout(dq)
        else:
            q, k, v, out, go = (t.contiguous() for t in (q, k, v, out, grad_output))
            dq, dk, dv = (torch.empty(m.head_shape, dtype=torch.float32, device=dev) for _ in range(3))
        # in place of the ABI's two [NB*nnz] scratch arguments (models/attention_blockcuda.py:83-84)
        scratch = _scratch(m, ctx.index, True, dev)
        _lib.core().spion_attn_backward_scratch(
            m.attn_handle, q.data_ptr(), k.data_ptr(), v.data_ptr(), p_flat.data_ptr(), out.data_ptr(), go.data_ptr(),
            dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), *ctx.index.tail[:2], ctx.index.nnz, m.num_heads,
            _address(lin), _address(lout), _address(lgrad), *scratch[1:])
        _lib.check_error("attn_backward")
        return dq, dk, dv, None, None, None


def _address(layout):
    return None if layout is None else ctypes.addressof(layout)


def _scratch(m, index, backward, device):
    """Scratch of a call of the core: (tensor, pointer, floats).  Where there is no memory for it, what the element kernels, or
    the handle's workspaces, do with."""
    floats = _lib.core().spion_attn_scratch(m.attn_handle, *index.tail[:2], index.nnz, int(backward))
    if floats < 0:
        _lib.check_error("attn_backward" if backward else "attn_forward")
    least = max(m.num_batches * index.nnz, 1) if backward else 0
    try:
        t = torch.empty(max(floats, 0), dtype=torch.float32, device=device)
    except torch.cuda.OutOfMemoryError:
        if floats <= least:
            raise
        t = torch.empty(least, dtype=torch.float32, device=device)
    return (t, t.data_ptr(), t.numel()) if t.numel() else (None, None, 0)


def _empty_heads(shape, interleaved, device):
    """Uninitialised [B,H,L,d] tensor; ``interleaved``: in memory [B,L,H,d], i.e. [B,L,H*d] once the heads are merged."""
    B, H, L, d = shape
    if interleaved:
        return torch.empty((B, L, H, d), dtype=torch.float32, device=device).transpose(1, 2)
    return torch.empty(shape, dtype=torch.float32, device=device)


class _BlockAttentionBase(nn.Module):
    with_mask = False

    def __init__(self, config, attn_cpp, attn_handle):
        super().__init__()
        if attn_cpp is None or not attn_handle:
            raise _lib.SpionLibraryError(
                f"{type(self).__name__} needs the loaded HIP library and a handle from its init(); "
                "there is no fallback implementation"
            )
        self.emb_dim = config["head_dim"]
        self.num_heads = config["num_head"]
        self.seq_len = config["max_seq_len"]
        self.batch_size = config["batch_size"]
        self.block_size = config["block_size"]
        self.num_batches = self.batch_size * self.num_heads
        self.num_blocks = int(self.seq_len / self.block_size)
        self.attn_cpp = attn_cpp
        self.attn_handle = attn_handle
        self.csr_cache = CsrCache(handle=attn_handle)
        self.attn_func = _BlockAttnFunction
        self.head_shape = (self.batch_size, self.num_heads, self.seq_len, self.emb_dim)
        _lib.core().spion_use_output_cache(attn_handle, 0)  # the backward is handed the output instead
        # every kernel family (tile, hybrid, element) reads [B,H,L,d] views of projections in place
        self.reads_views = self.emb_dim in (16, 32, 64, 128)


    def key_operand(self, mask):
        """What the compiled node takes for the key mask: (mask, True) when the kernels read it themselves, (penalties
        [B, H*L], False) for a mask of another type or layout, (None, False) without one."""
        if not self.with_mask:
            return None, False
        if mask.dtype == torch.float32 and mask.is_cuda and mask.is_contiguous() and not mask.requires_grad \
                and mask.shape == (self.batch_size, self.seq_len):
            return mask, True
        return (1e6 * (1.0 - mask.repeat(1, self.num_heads))).to(torch.float32).contiguous(), False

    def run(self, query, key, value, mask, mat):
        """(out, p_flat) through the compiled autograd node (csrc/autograd_node.cpp) -- the same steps as
        ``_BlockAttnFunction`` with the node, the saved tensors and the allocations on the C++ side of PyTorch, which
        takes a forward + backward of the L = 1024 tasks from 0.10 to 0.05 ms of host time -- or through the Python
        function when SPION_PY_NODE=1."""
        node = _lib.autograd_node()
        if node is None:
            return self.attn_func.apply(query, key, value, mask, mat, self)
        if query.shape != self.head_shape:
            raise ValueError(f"query shape {tuple(query.shape)} does not match the handle {self.head_shape}")
        idx = self.csr_cache.get(mat, self.block_size)
        key_mask, is_mask = self.key_operand(mask)
        index = query.device.index
        try:
            out, p_flat = node.sparse_attention(query, key, value, key_mask, is_mask, idx.offsets, idx.columns,
                                                idx.sum_mat, self.attn_handle, idx.nnz, self.num_heads, self.reads_views,
                                                _lib._raw_stream(torch.cuda.current_device() if index is None else index))
        except RuntimeError as e:
            if str(e).startswith(("attn_forward:", "attn_backward:")):
                raise _lib.SpionLibraryError(str(e)) from None
            raise
        return out, p_flat


class CUDABlockAttention(_BlockAttentionBase):
    with_mask = False

    def forward(self, query, key, value, mask, mat):
        return self.run(query, key, value, mask, mat)
