"""The passes of the dense backward beside the walk that does without them in the caller's scratch (head dimension 32; on a GPU
only)."""
import ctypes

import pytest
import torch

from spion_amd import _lib
from tests.test_gpu_dense_groups import _heads, _module

pytestmark = pytest.mark.gpu


def _forward(B, H, L, layout, masked, operands, mask):
    """The module, and what a backward on its handle takes: q, k, v, the map key-major, out, dO in out's layout"""
    mod, cpp = _module(B, H, L, 32, masked)
    q, k, v, do = operands
    with torch.no_grad():
        out, p = mod(q, k, v, mask)
    p = p.transpose(2, 3)
    assert p.is_contiguous()
    return mod, cpp, (q, k, v, p, out, torch.empty_like(out).copy_(do))


def _call(mod, tensors, grads, *scratch):
    """The strided backward of C callers, in scratch if there is one"""
    core, q, out = _lib.core(), tensors[0], tensors[4]
    core.spion_set_stream(mod.attn_handle, torch.cuda.current_stream().cuda_stream)
    layouts = [_lib.head_layout(t) for t in (q, out, grads[0])]
    entry = core.spion_dense_backward_scratch if scratch else core.spion_dense_backward_strided
    entry(mod.attn_handle, *(t.data_ptr() for t in tensors), *(t.data_ptr() for t in grads), q.shape[1],
          *(ctypes.addressof(y) for y in layouts), *scratch)
    _lib.check_error("backward")


def test_a_recorded_backward_without_scratch_after_a_first_one_with_it():
    B, H, L, core = 50, 2, 288, _lib.core()
    gen = torch.Generator(device="cuda").manual_seed(4)
    mod, cpp, t = _forward(B, H, L, "plain", False, _heads(B, H, L, 32, "plain", 4, gen), torch.ones(B, L, device="cuda"))
    floats = core.spion_dense_scratch(mod.attn_handle)
    scratch = torch.empty(max(floats, 1), device="cuda")
    first = [torch.empty_like(t[0]) for _ in range(3)]
    _call(mod, t, first, scratch.data_ptr(), floats)
    grads = [torch.empty_like(t[0]) for _ in range(3)]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        _call(mod, t, grads)
    passes = [torch.empty_like(t[0]) for _ in range(3)]
    for _ in range(3):
        for x in grads:
            x.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        _call(mod, t, passes)
        torch.cuda.synchronize()
        assert all(torch.equal(x, y) for x, y in zip(grads, passes))
    cpp.destroy(mod.attn_handle)
