"""The compiled autograd node (spion_amd/csrc/autograd_node.cpp) against the Python function it mirrors
(spion_amd/attention_blockcuda.py, itself the counterpart of models/attention_blockcuda.py:20-112): both hand the same
tensors to the same entry points, so outputs, probabilities and gradients must agree bit for bit -- on contiguous
heads, on views of projections, on slices of a fused projection, with the key mask, and on an element pattern (whose
backward needs the dS scratch)."""
import numpy as np
import pytest
import torch

import spion_amd
from spion_amd import _lib, workloads
from spion_amd.attention import Attention
from spion_amd.attention_blockbf16 import _BlockBF16Function

pytestmark = pytest.mark.gpu


def _module(B, H, L, d, bs, with_mask):
    cfg = dict(head_dim=d, num_head=H, max_seq_len=L, batch_size=B, block_size=bs)
    if with_mask:
        cpp = Attention._blockcuda_mask_compile_module()
        return spion_amd.CUDABlockMaskAttention(cfg, cpp, cpp.init(d, L, B * H, bs)), cpp
    cpp = Attention._blockcuda_compile_module()
    return spion_amd.CUDABlockAttention(cfg, cpp, cpp.init(d, L, B * H, bs)), cpp


def _inputs(B, H, L, d, layout, seed):
    g = torch.Generator().manual_seed(seed)
    if layout == "contiguous":
        q, k, v = (torch.randn(B, H, L, d, generator=g).cuda() for _ in range(3))
    elif layout == "proj":  # [B, L, H*d] projections viewed as heads
        q, k, v = (torch.randn(B, L, H, d, generator=g).cuda().transpose(1, 2) for _ in range(3))
    else:  # slices of one [B, L, 3, H, d] projection
        buf = torch.randn(B, L, 3, H, d, generator=g).cuda()
        q, k, v = (buf[:, :, i].transpose(1, 2) for i in range(3))
    do = torch.randn(B, H, L, d, generator=g).cuda()
    return q, k, v, do


@pytest.mark.parametrize("layout", ["contiguous", "proj", "fused"])
@pytest.mark.parametrize("with_mask", [False, True])
@pytest.mark.parametrize("pattern", ["tile", "element"])
def test_node_equals_python_function(layout, with_mask, pattern):
    node = _lib.autograd_node()
    if node is None:
        pytest.skip("SPION_PY_NODE=1: the Python function is the only path in this process")
    B, H, L, d = 2, 2, 256, 32
    if pattern == "tile":
        bs = 32
        mat_np = workloads.band_random_block_mask(L // bs, 1, extra_frac=0.1, seed=3).astype(np.float32)
    else:
        bs = 1
        sm, off, col = workloads.window_random_csr(L, 40, 100, seed=3)
        mat_np = np.zeros((L, L), dtype=np.float32)
        mat_np[np.repeat(np.arange(L), sm), col] = 1.0
    mat = torch.from_numpy(mat_np).cuda()
    mod, cpp = _module(B, H, L, d, bs, with_mask)
    key_mask = workloads.valid_length_mask(B, L, L // 2, L, seed=5).cuda() if with_mask else torch.ones(B, L, device="cuda")
    results = []
    for use_node in (True, False):
        q, k, v, do = _inputs(B, H, L, d, layout, seed=11)  # the same values in fresh buffers of the same layout
        leaves = [q, k, v]
        for t in leaves:
            t.requires_grad_()
        if use_node:
            out, p = mod.run(*leaves, key_mask, mat)
        else:
            out, p = mod.attn_func.apply(*leaves, key_mask, mat, mod)
        gq, gk, gv = torch.autograd.grad(out, leaves, do)
        torch.cuda.synchronize()
        results.append((out.detach(), p.detach(), gq, gk, gv))
        if layout == "fused":  # the gradients come back as slices of one buffer in both cases
            assert _lib.adjacent_head_views(gq, gk, gv)
    for a, b, name in zip(results[0], results[1], ("out", "p", "dq", "dk", "dv")):
        assert a.shape == b.shape and a.stride() == b.stride(), name
        assert torch.equal(a, b), name
    cpp.destroy(mod.attn_handle)


def test_node_ignores_the_gradient_of_the_probabilities_and_reports_errors():
    node = _lib.autograd_node()
    if node is None:
        pytest.skip("SPION_PY_NODE=1")
    B, H, L, d, bs = 1, 2, 128, 32, 32
    mat = torch.from_numpy(workloads.band_random_block_mask(L // bs, 1, extra_frac=0.2, seed=1).astype(np.float32)).cuda()
    mod, cpp = _module(B, H, L, d, bs, False)
    ones = torch.ones(B, L, device="cuda")
    q, k, v, do = _inputs(B, H, L, d, "contiguous", seed=2)
    for t in (q, k, v):
        t.requires_grad_()
    out, p = mod(q, k, v, ones, mat)
    # only the probabilities are used downstream: their gradient is ignored, the inputs get the gradient of a zero dO
    (p.sum() + 0.0 * out.sum()).backward()
    assert torch.count_nonzero(q.grad) == 0 and torch.count_nonzero(k.grad) == 0 and torch.count_nonzero(v.grad) == 0
    with pytest.raises(ValueError):
        mod(q[:, :1], k[:, :1], v[:, :1], ones, mat)
    cpp.destroy(mod.attn_handle)


@pytest.mark.parametrize("which", ["query", "key", "value", "mask"])
def test_forward_mode_is_refused_also_without_gradients(which):
    """Forward-mode AD does not depend on grad mode: a tangent must not be dropped because the node is passed by."""
    import torch.autograd.forward_ad as fwd

    if _lib.autograd_node() is None:
        pytest.skip("SPION_PY_NODE=1")
    B, H, L, d, bs = 1, 2, 64, 32, 32
    mat = torch.eye(L // bs, device="cuda")
    mod, cpp = _module(B, H, L, d, bs, True)
    q, k, v, _ = _inputs(B, H, L, d, "contiguous", seed=2)
    ones = torch.ones(B, L, device="cuda")
    args = dict(query=q, key=k, value=v, mask=ones)
    for guard in (torch.no_grad(), torch.enable_grad()):
        with guard, fwd.dual_level():
            dual = dict(args, **{which: fwd.make_dual(args[which], torch.ones_like(args[which]))})
            with pytest.raises(RuntimeError, match="jvp"):
                mod(dual["query"], dual["key"], dual["value"], dual["mask"], mat)
    with torch.no_grad(), fwd.dual_level():  # no tangent among the inputs
        mod(q, k, v, ones, mat)
    cpp.destroy(mod.attn_handle)


@pytest.mark.parametrize("which", ["input", "weight", "bias"])
def test_forward_mode_is_refused_by_the_whole_layer_without_gradients(which):
    import torch.autograd.forward_ad as fwd

    if _lib.autograd_node() is None:
        pytest.skip("SPION_PY_NODE=1")
    B, L = 2, 64
    cfg = dict(head_dim=32, num_head=2, max_seq_len=L, batch_size=B, block_size=32, transformer_dim=64, attention_dropout=0.0,
               task="lra-image")
    layer = Attention(cfg, inference=True).cuda()
    layer.reconstruct_for_blocksparse(cfg)
    x, mat = torch.randn(B, L, 64, device="cuda"), torch.eye(2, device="cuda")
    with torch.no_grad(), fwd.dual_level():
        if which == "input":
            x = fwd.make_dual(x, torch.ones_like(x))
        else:
            t = getattr(layer.ff, which).detach()
            delattr(layer.ff, which)
            setattr(layer.ff, which, fwd.make_dual(t, torch.ones_like(t)))
        with pytest.raises(RuntimeError, match="jvp"):
            layer(x, torch.ones(B, L, device="cuda"), mat)


def test_projections_around_a_differentiable_core_are_twice_differentiable():
    """The layer with the plain PyTorch core: gradients of a function of the first gradients, against the same layer written
    out in float64.  Both routes are chains of fp32 products of at most 64 terms with values of order one: 2^-24 a step,
    some hundred steps in all."""
    B, H, L, d, dim = 2, 2, 32, 32, 64
    cfg = dict(head_dim=d, num_head=H, max_seq_len=L, batch_size=B, block_size=32, transformer_dim=dim, attention_dropout=0.0,
               task="lra-pathfinder32-curv_contour_length_14")
    torch.manual_seed(3)
    layer = Attention(cfg).cuda()
    mask = torch.ones(B, L, device="cuda")
    x, dy = torch.randn(B, L, dim, device="cuda", requires_grad=True), torch.randn(B, L, dim, device="cuda", requires_grad=True)
    params = list(layer.parameters())
    r = [torch.randn_like(t) for t in [x] + params]

    def written_out(x, dy, params):
        (wq, bq, wk, bk, wv, bv, wf, bf), lin = params, torch.nn.functional.linear
        q, k, v = (layer.split_heads(lin(x, w, b)) for w, b in ((wq, bq), (wk, bk), (wv, bv)))
        p = torch.softmax(q @ k.transpose(-1, -2) / d ** 0.5, -1)
        return lin(layer.combine_heads(p @ v), wf, bf)

    def second(forward, x, dy, params, r):
        first = torch.autograd.grad(forward(x, dy, params), [x] + params, dy, create_graph=True)
        return torch.autograd.grad(sum((a * b).sum() for a, b in zip(first, r)), [x, dy] + params, allow_unused=True)

    assert [n for n, _ in layer.named_parameters()] == [f"{m}.{t}" for m in ("W_q", "W_k", "W_v", "ff") for t in ("weight", "bias")]
    got = second(lambda x, dy, p: layer(x, mask)[0], x, dy, params, r)
    up = lambda t: t.detach().cpu().double().requires_grad_()
    ref = second(written_out, up(x), up(dy), [up(t) for t in params], [t.cpu().double() for t in r])
    assert len(got) == len(ref) == 10
    for a, b in zip(got, ref):
        if b is None or float(b.norm()) < 1e-9:  # (exactly zero: what a bias's shift leaves unchanged)
            assert a is None or float(a.norm()) < 1e-3
            continue
        assert float((a.cpu().double() - b).norm() / b.norm()) < 1e-5


# ---- the dense-phase modules and the bf16 module ---------------------------------------------------
def _python_only(mod, fn):
    mod._node_takes = lambda *a: False
    try:
        return fn()
    finally:
        del mod._node_takes


@pytest.mark.parametrize("layout", ["contiguous", "proj", "fused", "mixed"])
@pytest.mark.parametrize("mask_kind", [None, "float", "double"])
@pytest.mark.parametrize("d", [32, 64])
def test_dense_node_equals_python_function(layout, mask_kind, d):
    if _lib.autograd_node() is None:
        pytest.skip("SPION_PY_NODE=1")
    B, H, L = 2, 2, 160
    cfg = dict(head_dim=d, num_head=H, max_seq_len=L, batch_size=B)
    cpp = getattr(Attention, "_cuda_mask_compile_module" if mask_kind else "_cuda_compile_module")()
    mod = (spion_amd.CUDAMaskAttention if mask_kind else spion_amd.CUDAAttention)(cfg, cpp, cpp.init(d, L, B * H))
    mask = workloads.valid_length_mask(B, L, L // 2, L, seed=5).cuda()
    if mask_kind == "double":  # the penalties are then made by torch
        mask = mask.double()

    def step(grad):
        leaves = [t.requires_grad_(grad) for t in _inputs(B, H, L, d, layout if layout != "mixed" else "contiguous", seed=11)[:3]]
        do = _inputs(B, H, L, d, "contiguous", seed=12)[3]
        if layout == "mixed":  # no common strides: copies
            leaves[1] = leaves[1].detach().transpose(1, 2).contiguous().transpose(1, 2).requires_grad_(grad)
        mod.score_map = None
        with torch.set_grad_enabled(grad):
            out, attn = mod(*leaves, mask)
        grads = torch.autograd.grad(out, leaves, do) if grad else ()
        if grad and layout == "fused":
            assert _lib.adjacent_head_views(*grads)
        return [out.detach(), attn.detach(), *grads] + ([mod.score_map] if mod.emit_score_map else [])

    for emit in (False, True):
        mod.emit_score_map = emit
        for grad in (True, False):
            a, b = step(grad), _python_only(mod, lambda: step(grad))
            assert len(a) == len(b) and all(x.stride() == y.stride() and torch.equal(x, y) for x, y in zip(a, b))
    cpp.destroy(mod.attn_handle)


@pytest.mark.parametrize("layout", ["contiguous", "proj", "mixed"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("mask_kind", [None, "float", "double"])
def test_bf16_node_equals_python_function(layout, dtype, mask_kind):
    if _lib.autograd_node() is None:
        pytest.skip("SPION_PY_NODE=1")
    B, H, L, d, bs = 2, 2, 256, 64, 32
    mod = spion_amd.BlockAttentionBF16(dict(head_dim=d, num_head=H, max_seq_len=L, batch_size=B, block_size=bs), mask_kind is not None)
    mat = torch.from_numpy(workloads.band_random_block_mask(L // bs, 1, extra_frac=0.1, seed=3).astype(np.float32)).cuda()
    mask = workloads.valid_length_mask(B, L, L // 2, L, seed=5).cuda()
    if mask_kind == "double":
        mask = mask.double()

    def step(grad):
        leaves = [t.to(dtype).requires_grad_(grad) for t in _inputs(B, H, L, d, "contiguous" if layout == "mixed" else layout, seed=11)[:3]]
        if layout == "mixed":
            leaves[1] = leaves[1].detach().transpose(1, 2).contiguous().transpose(1, 2).requires_grad_(grad)
        with torch.set_grad_enabled(grad):
            out, zero = mod(*leaves, mask, mat)
        assert zero == 0
        do = _inputs(B, H, L, d, "contiguous", seed=12)[3].to(torch.bfloat16)
        return [out.detach()] + (list(torch.autograd.grad(out, leaves, do)) if grad else [])

    for grad in (True, False):
        a, b = step(grad), _python_only(mod, lambda: step(grad))
        assert len(a) == len(b) and all(x.dtype == y.dtype and x.stride() == y.stride() and torch.equal(x, y) for x, y in zip(a, b))
    mod.lib.spion_block_bf16_destroy(mod.attn_handle)


def test_dense_and_bf16_nodes_leave_other_calls_to_the_python_functions():
    """Wrong sizes and types keep their errors, forward mode stays refused, the map's gradient is ignored."""
    import torch.autograd.forward_ad as fwd

    if _lib.autograd_node() is None:
        pytest.skip("SPION_PY_NODE=1")
    B, H, L, d = 1, 2, 64, 32
    cfg = dict(head_dim=d, num_head=H, max_seq_len=L, batch_size=B, block_size=32)
    cpp = Attention._cuda_compile_module()
    dense = spion_amd.CUDAAttention(cfg, cpp, cpp.init(d, L, B * H))
    bf16 = spion_amd.BlockAttentionBF16(cfg)
    q, k, v, _ = _inputs(B, H, L, d, "contiguous", seed=2)
    ones, mat = torch.ones(B, L, device="cuda"), torch.ones(2, 2, device="cuda")
    half = [t.bfloat16() for t in (q, k, v)]
    with pytest.raises(ValueError):
        dense(q[:, :1], k[:, :1], v[:, :1], ones)
    with pytest.raises(ValueError):
        bf16(half[0], half[1][:, :, :32], half[2], ones, mat)
    for guard in (torch.no_grad(), torch.enable_grad()):
        with guard, fwd.dual_level():
            with pytest.raises(RuntimeError, match="jvp"):
                dense(q, fwd.make_dual(k, torch.ones_like(k)), v, ones)
            with pytest.raises(RuntimeError, match="jvp"):
                bf16(fwd.make_dual(half[0], torch.ones_like(half[0])), half[1], half[2], ones, mat)
    leaves = [t.clone().requires_grad_() for t in (q, k, v)]
    out, attn = dense(*leaves, ones)
    (attn.sum() + 0.0 * out.sum()).backward()
    assert all(torch.count_nonzero(t.grad) == 0 for t in leaves)
    cpp.destroy(dense.attn_handle)
    bf16.lib.spion_block_bf16_destroy(bf16.attn_handle)


def _of_kind(kind, B, H, L, d):
    """(module, what its forward takes after the heads, destroy)"""
    cfg = dict(head_dim=d, num_head=H, max_seq_len=L, batch_size=B, block_size=32)
    ones, mat = torch.ones(B, L, device="cuda"), torch.ones(L // 32, L // 32, device="cuda")
    if kind == "dense":
        cpp = Attention._cuda_mask_compile_module()
        return spion_amd.CUDAMaskAttention(cfg, cpp, cpp.init(d, L, B * H)), (ones,), cpp.destroy
    if kind == "bf16":
        mod = spion_amd.BlockAttentionBF16(cfg, True)
        return mod, (ones, mat), mod.lib.spion_block_bf16_destroy
    mod, cpp = _module(B, H, L, d, 32, True)
    return mod, (ones, mat), cpp.destroy


def _layer(B, H, L, d):
    cfg = dict(head_dim=d, num_head=H, max_seq_len=L, batch_size=B, block_size=32, transformer_dim=H * d, attention_dropout=0.0,
               task="lra-text")
    mod = Attention(cfg, inference=True).cuda()
    mod.reconstruct_for_blocksparse(cfg)
    return mod


@pytest.mark.parametrize("kind", ["sparse", "dense", "bf16"])
def test_nodes_hold_their_handle_and_refuse_short_masks(kind):
    """The backward works on the module's handle: a graph that outlives its caller's module holds it, also where it is destroyed
    with the module, and lets it go.  A mask with fewer entries than [B, L], or on the host, is refused before a kernel reads
    past its end."""
    import gc
    import weakref

    if _lib.autograd_node() is None:
        pytest.skip("SPION_PY_NODE=1")
    B, H, L, d = 2, 2, 64, 32
    dtype = torch.bfloat16 if kind == "bf16" else torch.float32
    q, k, v, do = (t.to(dtype) for t in _inputs(B, H, L, d, "contiguous", seed=2))
    alive = _lib.core().spion_debug_handles()
    mod, (mask, *rest), destroy = _of_kind(kind, B, H, L, d)
    with pytest.raises(ValueError):
        mod(q, k, v, torch.ones(1, L, device="cuda"), *rest)
    with pytest.raises(RuntimeError):
        mod(q, k, v, torch.ones(B, L), *rest)
    leaves = [t.clone().requires_grad_() for t in (q, k, v)]
    want = torch.autograd.grad(mod(*leaves, mask, *rest)[0], leaves, do)
    gc.collect()
    weakref.finalize(mod, destroy, mod.attn_handle)
    held = weakref.ref(mod)
    out = mod(*leaves, mask, *rest)[0]
    del mod
    gc.collect()
    assert held() is None and _lib.core().spion_debug_handles() == alive + 1
    grads = torch.autograd.grad(out, leaves, do)
    assert all(torch.equal(a, b) for a, b in zip(grads, want))
    del out, grads
    gc.collect()
    assert _lib.core().spion_debug_handles() == alive


@pytest.mark.parametrize("kind", ["sparse", "sparse_plain", "dense", "dense_mean", "bf16", "layer"])
def test_compiled_autograd_takes_the_nodes(kind):
    """A recorded graph's backward through torch's compiled autograd: the gradients of the plain one, bit for bit."""
    from torch._dynamo import compiled_autograd

    B, H, L, d = 2, 2, 64, 32
    dtype = torch.bfloat16 if kind == "bf16" else torch.float32
    *leaves, do = (t.to(dtype) for t in _inputs(B, H, L, d, "contiguous", seed=2))
    ones, mat = torch.ones(B, L, device="cuda"), torch.ones(2, 2, device="cuda")
    destroy = None
    if kind == "layer":
        mod, rest = _layer(B, H, L, d), (ones, mat)
        leaves, do = [leaves[0].transpose(1, 2).reshape(B, L, H * d)], do.transpose(1, 2).reshape(B, L, H * d)
    elif kind == "sparse_plain":
        (mod, cpp), rest = _module(B, H, L, d, 32, False), (ones, mat)
        destroy = cpp.destroy
    else:
        mod, rest, destroy = _of_kind(kind.removesuffix("_mean"), B, H, L, d)
        mod.emit_score_map = kind == "dense_mean"
    leaves = [t.requires_grad_() for t in leaves]
    want = torch.autograd.grad(mod(*leaves, *rest)[0], leaves, do)
    out, second = mod(*leaves, *rest)
    if isinstance(second, torch.Tensor) and kind == "sparse":
        assert not second.requires_grad
    with compiled_autograd._enable(torch.compile(backend="eager")):
        out.backward(do)
    assert all(torch.equal(a, t.grad) for a, t in zip(want, leaves))
    if kind == "dense_mean":
        assert not mod.score_map.requires_grad
    if destroy:
        destroy(mod.attn_handle)


@pytest.mark.parametrize("kind", ["sparse", "dense", "bf16", "layer"])
def test_backward_runs_on_the_callers_stream(kind):
    """A forward on a side stream, its node called on another, where the gradient is only just being made (by the node itself;
    for the layer's three nodes by compiled autograd, which does not go back to the forward's stream either)."""
    from torch._dynamo import compiled_autograd

    if _lib.autograd_node() is None:
        pytest.skip("SPION_PY_NODE=1")
    B, H, L, d = 2, 2, 64, 32
    dtype = torch.bfloat16 if kind == "bf16" else torch.float32
    *leaves, do = (t.to(dtype) for t in _inputs(B, H, L, d, "contiguous", seed=3))
    destroy = None
    if kind == "layer":
        mod, rest = _layer(B, H, L, d), (torch.ones(B, L, device="cuda"), torch.ones(2, 2, device="cuda"))
        leaves, do = [leaves[0].transpose(1, 2).reshape(B, L, H * d)], do.transpose(1, 2).reshape(B, L, H * d)
    else:
        mod, rest, destroy = _of_kind(kind, B, H, L, d)
    leaves = [t.requires_grad_() for t in leaves]
    want = torch.autograd.grad(mod(*leaves, *rest)[0], leaves, do)
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        out = mod(*leaves, *rest)[0]
    torch.cuda.synchronize()
    late = torch.full_like(do, float("nan"))
    torch.cuda._sleep(20_000_000)
    late.copy_(do)
    if kind == "layer":
        with compiled_autograd._enable(torch.compile(backend="eager")):
            out.backward(late)
        got = [t.grad for t in leaves]
    else:
        got = out.grad_fn(late, None) if kind == "dense" else out.grad_fn(late)
    assert all(torch.equal(a, b) for a, b in zip(want, got))
    if destroy:
        destroy(mod.attn_handle)


@pytest.mark.parametrize("kind", ["sparse", "dense", "bf16"])
def test_modules_that_keep_their_outputs_are_collected(kind):
    import gc
    import weakref

    B, H, L, d = 2, 2, 64, 32
    q, k, v, do = (t.to(torch.bfloat16 if kind == "bf16" else torch.float32) for t in _inputs(B, H, L, d, "contiguous", seed=2))
    alive = _lib.core().spion_debug_handles()
    for backward in (False, True):
        mod, rest, destroy = _of_kind(kind, B, H, L, d)
        weakref.finalize(mod, destroy, mod.attn_handle)
        freed = weakref.ref(mod)
        mod.kept = mod(*(t.clone().requires_grad_() for t in (q, k, v)), *rest)[0]
        if backward:
            mod.kept.backward(do)
        del mod
        gc.collect()
        assert freed() is None and _lib.core().spion_debug_handles() == alive


@pytest.mark.parametrize("kind", ["sparse", "dense", "bf16"])
def test_python_functions_refuse_other_types_and_masks(kind):
    """Heads in another type (those of bf16 are converted), and masks short or on the host, which kernels would read past
    their end."""
    B, H, L, d = 2, 2, 64, 32
    mod, (ones, *rest), destroy = _of_kind(kind, B, H, L, d)
    function = _BlockBF16Function if kind == "bf16" else mod.attn_func
    q, k, v, _ = _inputs(B, H, L, d, "contiguous", seed=2)
    with torch.no_grad():
        function.apply(q, k, v, ones, *rest, mod)
        for heads in ((q.half(), k, v), (q, k, v.half())) if kind != "bf16" else ():
            with pytest.raises(RuntimeError, match="fp32"):
                function.apply(*heads, ones, *rest, mod)
            with pytest.raises(RuntimeError, match="fp32"):
                mod(*heads, ones, *rest)
        with pytest.raises(ValueError, match="key mask"):
            function.apply(q, k, v, ones[:1], *rest, mod)
        with pytest.raises(RuntimeError, match="one GPU"):
            function.apply(q, k, v, ones.cpu(), *rest, mod)
        with pytest.raises(RuntimeError, match="one GPU"):
            function.apply(q, k.cpu(), v, ones, *rest, mod)
    destroy(mod.attn_handle)


@pytest.mark.parametrize("python", [False, True])
@pytest.mark.parametrize("kind", ["sparse", "bf16"])
def test_saved_tensor_hooks_do_not_meet_the_index(kind, python):
    """The library knows an index by its address: one that a hook brings back somewhere else would be analysed again, and
    stay on file for whatever index comes to lie there next.  Masks of as many entries taken in turn, everything saved moved
    to the host: the gradients as without, bit for bit, and the hooks see floating tensors alone."""
    B, H, L, d = 2, 2, 128, 32
    mod, (ones, _), destroy = _of_kind(kind, B, H, L, d)
    dtype = torch.bfloat16 if kind == "bf16" else torch.float32
    *leaves, do = (t.to(dtype) for t in _inputs(B, H, L, d, "contiguous", seed=6))
    leaves = [t.requires_grad_() for t in leaves]
    mats = [torch.eye(4, device="cuda").roll(k, 0).contiguous() for k in range(3)]
    seen = set()

    def pack(t):
        seen.add(t.dtype)
        return t.cpu()

    def forward(m):
        if not python:
            return mod(*leaves, ones, m)[0]
        if kind == "bf16":
            return _BlockBF16Function.apply(*leaves, ones, m, mod)
        return mod.attn_func.apply(*leaves, ones, m, mod)[0]

    want = [torch.autograd.grad(forward(m), leaves, do) for m in mats]
    for m, w in list(zip(mats, want)) * 2:
        with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.cuda()):
            out = forward(m)
        got = torch.autograd.grad(out, leaves, do)
        assert all(torch.equal(a, b) for a, b in zip(got, w))
    assert all(t.is_floating_point for t in seen)
    destroy(mod.attn_handle)


@pytest.mark.parametrize("python", [False, True])
@pytest.mark.parametrize("kind", ["sparse", "dense", "bf16", "layer"])
@pytest.mark.parametrize("layout", ["contiguous", "proj", "fused"])
def test_saved_tensors_that_hooks_change_one_by_one(kind, python, layout):
    """One saved tensor at a time: in other strides the gradients are the same bits; on the host, of another type or size it
    is refused.  (Key penalties, which the bf16 node saves last, may be more than the heads need.)"""
    if not python and _lib.autograd_node() is None:
        pytest.skip("SPION_PY_NODE=1")
    if kind == "layer" and (python or layout != "contiguous"):
        pytest.skip("the whole layer in one call has one form")
    B, H, L, d = 2, 2, 64, 32
    dtype = torch.bfloat16 if kind == "bf16" else torch.float32
    *leaves, do = _inputs(B, H, L, d, layout, seed=4)
    leaves, do = [t.to(dtype).requires_grad_() for t in leaves], do.to(dtype)
    if kind == "layer":
        mod, rest, destroy = _layer(B, H, L, d), (torch.ones(B, L, device="cuda"), torch.ones(L // 32, L // 32, device="cuda")), None
        leaves, do = [leaves[0].detach().transpose(1, 2).reshape(B, L, H * d).requires_grad_()], do.reshape(B, L, H * d)
    else:
        mod, rest, destroy = _of_kind(kind, B, H, L, d)
    function = _BlockBF16Function if kind == "bf16" else getattr(mod, "attn_func", None)

    def step(which, change):
        packed = []

        def pack(t):
            packed.append(t)
            return len(packed) - 1

        with torch.autograd.graph.saved_tensors_hooks(pack, lambda i: change(packed[i]) if i == which else packed[i]):
            out = function.apply(*leaves, *rest, mod) if python else mod(*leaves, *rest)
        grads = torch.autograd.grad(out if isinstance(out, torch.Tensor) else out[0], leaves, do)
        return len(packed), grads

    n, want = step(-1, None)
    assert n == (11 if kind == "layer" else 5 + (kind == "bf16" and not python))
    interleaved = lambda t: t.transpose(-3, -2).contiguous().transpose(-3, -2) if t.dim() == 4 else t.clone()
    for i in range(n):
        for change in (torch.Tensor.contiguous, interleaved, lambda t: torch.stack([t, t], -1)[..., 0]):
            assert all(torch.equal(a, b) for a, b in zip(step(i, change)[1], want))
        for change in (torch.Tensor.cpu, torch.Tensor.double, lambda t: t[:1].clone() if t.dim() > 1 else t[:1]):
            with pytest.raises(TypeError):
                step(i, change)
    if destroy:
        destroy(mod.attn_handle)


def test_nodes_refuse_heads_the_strided_entries_cannot_take():
    """Contiguous heads off 16 bytes, and saved heads that hooks bring back so: refused as by the Python functions.  Hooks
    that bring them back contiguous change nothing."""
    if _lib.autograd_node() is None:
        pytest.skip("SPION_PY_NODE=1")
    B, H, L, d = 2, 2, 64, 32
    cfg = dict(head_dim=d, num_head=H, max_seq_len=L, batch_size=B, block_size=32)
    cpp = Attention._cuda_compile_module()
    dense = spion_amd.CUDAAttention(cfg, cpp, cpp.init(d, L, B * H))
    bf16 = spion_amd.BlockAttentionBF16(cfg)
    ones, mat = torch.ones(B, L, device="cuda"), torch.ones(2, 2, device="cuda")

    def off(t):
        return torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape)

    q, k, v, do = _inputs(B, H, L, d, "proj", seed=4)
    for call in (lambda: dense(off(q), k, v, ones), lambda: _python_only(dense, lambda: dense(off(q), k, v, ones))):
        with pytest.raises(TypeError):
            call()
    for mod, rest, t in ((dense, (ones,), (q, k, v)), (bf16, (ones, mat), tuple(x.bfloat16() for x in (q, k, v)))):
        leaves = [x.clone(memory_format=torch.preserve_format).requires_grad_() for x in t]

        def step(unpack):
            with torch.autograd.graph.saved_tensors_hooks(lambda x: x, unpack):
                out = mod(*leaves, *rest)[0]
            return torch.autograd.grad(out, leaves, do.to(out.dtype))

        for a, b in zip(step(lambda x: x), step(lambda x: x.contiguous())):
            assert torch.equal(a, b)
        with pytest.raises(TypeError):
            step(off)
    cpp.destroy(dense.attn_handle)
    bf16.lib.spion_block_bf16_destroy(bf16.attn_handle)


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("kind", ["sparse", "sparse_mask", "dense", "dense_mask", "bf16", "layer"])
def test_traced_modules_compute(kind, grad):
    """torch.jit.trace records the modules' Python functions: a traced module gives on other inputs what the module gives,
    with gradients.  (The layer's projections are torch's products then: 1e-5 of the 2-norm.)"""
    B, H, L, d = 2, 2, 64, 32
    cfg = dict(head_dim=d, num_head=H, max_seq_len=L, batch_size=B, block_size=32, transformer_dim=H * d, attention_dropout=0.0,
               task="lra-image")
    mask, mat = torch.ones(B, L, device="cuda"), torch.ones(2, 2, device="cuda")
    mask[0, L // 2:] = 0
    rest = (mask,) if kind.startswith("dense") else (mask, mat)
    if kind == "layer":
        mod = Attention(cfg, inference=True).cuda().requires_grad_(grad)
        mod.reconstruct_for_blocksparse(cfg)
    elif kind.startswith("dense"):
        cpp = getattr(Attention, "_cuda_mask_compile_module" if kind == "dense_mask" else "_cuda_compile_module")()
        cls = spion_amd.CUDAMaskAttention if kind == "dense_mask" else spion_amd.CUDAAttention
        mod = cls(cfg, cpp, cpp.init(d, L, B * H))
    elif kind == "bf16":
        mod = spion_amd.BlockAttentionBF16(cfg, True)
    else:
        mod, cpp = _module(B, H, L, d, 32, kind == "sparse_mask")

    class Caller(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.mod = mod

        def forward(self, *x):
            return 2 * self.mod(*x, *rest)[0]

    def inputs(seed):
        x = [torch.randn(B, L, H * d, generator=torch.Generator().manual_seed(seed)).cuda()] if kind == "layer" else \
            list(_inputs(B, H, L, d, "contiguous", seed)[:3])
        return [t.to(torch.bfloat16 if kind == "bf16" else t.dtype).requires_grad_(grad) for t in x]

    caller, x = Caller(), inputs(2)
    with torch.set_grad_enabled(grad):
        traced = torch.jit.trace(caller, tuple(inputs(1)), check_trace=False)
        got, want = [traced(*x)], [caller(*x)]
    if grad:
        go = torch.randn(want[0].shape, generator=torch.Generator().manual_seed(3)).to("cuda", want[0].dtype)
        got, want = (y + list(torch.autograd.grad(y[0], x, go)) for y in (got, want))
    for a, b in zip(got, want):
        assert float((a - b).norm()) <= 1e-5 * float(b.norm()) if kind == "layer" else torch.equal(a, b)
