"""Sizes the compiled node is handed are compared with the handle's before any kernel runs (the kernels take theirs from the
handle), and the layer leaves a call that does not fit to the modules' own errors.  Host code only: no kernel is launched."""
import pytest
import torch

import spion_amd
from spion_amd import _lib
from spion_amd.attention import Attention
from spion_amd.attention_blockbf16 import _BlockBF16Function

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


@needs_node
@pytest.mark.parametrize("is_mask", [True, False])
def test_node_refuses_a_key_mask_on_another_device(is_mask):
    """(No handle is looked at before.)"""
    node, q, index = _lib.autograd_node(), torch.zeros(2, 2, 64, 32), torch.zeros(4, dtype=torch.int32)
    mask = torch.zeros(2, 64, device="meta")
    weights = [torch.zeros(64, 64)] * 3 + [torch.zeros(64)] * 3 + [torch.zeros(64, 64), torch.zeros(64)]
    for call in (lambda: node.sparse_attention(q, q, q, mask, is_mask, index, index, index, 0, 1, 2, True, 0),
                 lambda: node.dense_attention(q, q, q, mask, is_mask, 0, False, 0),
                 lambda: node.bf16_attention(q, q, q, mask, is_mask, index, index, index, 0, 1, 0),
                 lambda: node.sparse_layer(torch.zeros(2, 64, 64), *weights, mask, is_mask, index, index, index, 0, 1, 2, 32, 0)):
        with pytest.raises(RuntimeError, match="one GPU"):
            call()


@pytest.mark.parametrize("family", ["sparse", "dense", "dense_feature_major", "bf16"])
@pytest.mark.parametrize("which", range(3))
def test_python_functions_refuse_what_the_handle_does_not_fit(family, which):
    """The Python functions, which take the calls that the compiled node leaves them and those under torch.jit.trace, check
    query, key and value: a key or value of fewer rows, a host tensor."""
    d, L = (64, 2080) if family == "dense_feature_major" else (32, 64)
    cfg = _config(2, d, L)
    mat, mask = torch.ones(2, 2), torch.ones(2, L)
    if family == "bf16":
        mod = spion_amd.BlockAttentionBF16(cfg)
        call = lambda *heads: _BlockBF16Function.apply(*heads, mask, mat, mod)
    elif family == "sparse":
        cpp = Attention._blockcuda_compile_module()
        mod = spion_amd.CUDABlockAttention(cfg, cpp, cpp.init(d, L, 4, 32))
        call = lambda *heads: mod.attn_func.apply(*heads, mask, mat, mod)
    else:
        cpp = Attention._cuda_compile_module()
        mod = spion_amd.CUDAAttention(cfg, cpp, cpp.init(d, L, 4))
        assert mod.reads_views == (family == "dense")
        call = lambda *heads: mod(*heads, mask)
    heads = [torch.zeros(2, 2, L, d) for _ in range(3)]
    with pytest.raises(RuntimeError, match="GPU expected"):
        call(*heads)
    heads[which] = heads[which][:, :, :32]
    with pytest.raises(ValueError, match="does not match the handle"):
        call(*heads)


class _Unused:
    def __getattr__(self, name):
        raise AssertionError(f"the compiled node's {name} was called")


@pytest.mark.parametrize("heads,d", [(4, 32), (1, 32), (2, 64), (1, 64), (4, 16)])
def test_layer_with_a_core_of_other_heads_is_not_taken_in_one_call(heads, d):
    """reconstruct_for_blocksparse has a config of its own: a core for other heads than the layer's."""
    layer = Attention(_config(2, 32), inference=True)
    layer.reconstruct_for_blocksparse(_config(heads, d))
    x = torch.zeros(2, 64, 64)
    assert layer._sparse_layer(_Unused(), (None,) * 8, x, torch.ones(2, 64), torch.ones(2, 2)) is None


def _linears(n, dim, out):
    w = [torch.zeros(n, dim) for _ in range(3)] + [torch.zeros(out, n)]
    return w, [torch.zeros(t.shape[0]) for t in w]


def _fits(x, w, b, heads=2, d=32):
    return _lib.autograd_node().projections_fit(x, w[0], w[1], w[2], b[0], b[1], b[2], w[3], b[3], heads, d)


@needs_node
def test_projections_fit_only_weights_of_the_layers_sizes():
    x = torch.zeros(2, 64, 96)
    assert _fits(x, *_linears(64, 96, 96))
    assert _fits(x, *_linears(64, 96, 128))  # an output projection to another width
    assert not _fits(x, *_linears(64, 96, 48))  # which is no multiple of 32
    assert not _fits(torch.zeros(2, 48, 96)[:1], *_linears(64, 96, 96))  # rows
    assert not _fits(torch.zeros(2, 64, 80), *_linears(64, 80, 96))  # features
    assert not _fits(torch.zeros(0, 64, 96), *_linears(64, 96, 96))
    assert not _fits(torch.zeros(64, 96), *_linears(64, 96, 96))
    for i in range(4):
        for bad in ((32, 96), (64, 64), (96, 64), (64, 160)):
            w, b = _linears(64, 96, 96)
            if tuple(w[i].shape) == bad or (i == 3 and bad[1] == 64):
                continue
            w[i] = torch.zeros(bad)
            assert not _fits(x, w, b), (i, bad)
        for bad in (torch.zeros(32), torch.zeros(64, 1), torch.zeros(64).double(), torch.zeros(64, device="meta")):
            w, b = _linears(64, 96, 96)
            b[i] = bad
            assert not _fits(x, w, b), (i, bad.shape, bad.dtype, bad.device)
        w, b = _linears(64, 96, 96)
        w[i] = w[i].half()
        assert not _fits(x, w, b)


@needs_node
@pytest.mark.parametrize("which", ["rows", "columns", "bias", "type"])
def test_node_refuses_projections_of_other_sizes(which):
    w, b = _linears(64, 96, 96)
    w[1] = {"rows": torch.zeros(32, 96), "columns": torch.zeros(64, 64), "type": torch.zeros(64, 96).double()}.get(which, w[1])
    b[1] = torch.zeros(32) if which == "bias" else b[1]
    with pytest.raises(ValueError, match="projection"):
        _lib.autograd_node().project_heads(torch.zeros(2, 64, 96), w[0], w[1], w[2], b[0], b[1], b[2], 2, 32, 0)
    with pytest.raises(ValueError, match="projection"):
        _lib.autograd_node().merge_heads(torch.zeros(2, 2, 64, 32 if which == "rows" else 48), torch.zeros(64, 96), torch.zeros(32), 0)


def test_bf16_module_reports_a_failed_key_penalty(monkeypatch):
    """The penalties' buffer is uninitialised where the launch failed: the call must not go on with it."""
    from types import SimpleNamespace

    from spion_amd import attention_blockbf16 as bf16

    monkeypatch.setattr(_lib, "_raw_stream", lambda index: 0)
    mask = SimpleNamespace(dtype=torch.float32, is_cuda=True, is_contiguous=lambda: True, shape=(2, 64), data_ptr=lambda: 0)
    m = SimpleNamespace(batch_size=2, seq_len=64, num_heads=2, num_batches=4, lib=_lib.core())
    dev = SimpleNamespace(index=0)
    monkeypatch.setattr(bf16.torch, "empty", lambda *a, **k: SimpleNamespace(data_ptr=lambda: 0))
    with pytest.raises(_lib.SpionLibraryError, match="spion_key_penalty"):
        bf16._penalty(mask, m, dev)
    monkeypatch.setattr(m, "lib", SimpleNamespace(spion_key_penalty=lambda *a: 1))
    with pytest.raises(_lib.SpionLibraryError, match="spion_key_penalty"):
        bf16._penalty(mask, m, dev)
