"""Sizes the compiled node is handed are compared with the handle's before any kernel runs (the kernels take theirs from the
handle), and the layer leaves a call that does not fit to the modules' own errors.  Host code only: no kernel is launched."""
import pytest
import torch

import spion_amd
from spion_amd import _lib
from spion_amd.attention import Attention

needs_node = pytest.mark.skipif(_lib.autograd_node() is None, reason="SPION_PY_NODE=1")


def _config(heads, d, L=64, B=2, task="lra-image", dim=64):
    return dict(head_dim=d, num_head=heads, max_seq_len=L, batch_size=B, block_size=32, transformer_dim=dim,
                attention_dropout=0.0, task=task)


@needs_node
@pytest.mark.parametrize("shape,heads", [((2, 1, 64, 64), 1), ((2, 4, 64, 32), 4), ((1, 2, 64, 32), 2), ((2, 2, 32, 32), 2),
                                         ((1, 4, 64, 32), 2), ((2, 2, 64, 64), 2)])
def test_node_refuses_heads_of_another_shape(shape, heads):
    """Batch, heads, length or head dimension other than the handle's (2 samples of 2 heads, 64 x 32), also where the number
    of elements or of heads in all is the same."""
    cpp = Attention._blockcuda_compile_module()
    handle = cpp.init(32, 64, 4, 32)
    q = torch.zeros(shape)
    index = torch.zeros(4, dtype=torch.int32)
    with pytest.raises(ValueError, match="does not match the handle"):
        _lib.autograd_node().sparse_attention(q, q, q, None, False, index, index, index, handle, 1, heads, True, 0)
    cpp.destroy(handle)


@needs_node
def test_node_refuses_a_key_mask_that_is_too_small():
    cpp = Attention._blockcuda_mask_compile_module()
    handle = cpp.init(32, 64, 4, 32)
    q = torch.zeros(2, 2, 64, 32)
    index = torch.zeros(4, dtype=torch.int32)
    with pytest.raises(ValueError, match="key mask"):
        _lib.autograd_node().sparse_attention(q, q, q, torch.zeros(2, 64), False, index, index, index, handle, 1, 2, True, 0)
    cpp.destroy(handle)


class _Unused:
    def __getattr__(self, name):
        raise AssertionError(f"the compiled node's {name} was called")


@pytest.mark.parametrize("heads,d", [(4, 32), (1, 32), (2, 64), (1, 64), (4, 16)])
def test_layer_with_a_core_of_other_heads_is_not_taken_in_one_call(heads, d):
    """reconstruct_for_blocksparse has a config of its own: a core for other heads than the layer's."""
    layer = Attention(_config(2, 32), inference=True)
    layer.reconstruct_for_blocksparse(_config(heads, d))
    x = torch.zeros(2, 64, 64)
    assert layer._sparse_layer(_Unused(), x, torch.ones(2, 64), torch.ones(2, 2)) is None
