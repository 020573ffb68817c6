"""The passes of the dense backward beside the walk that does without them in the caller's scratch (head dimension 32; on a GPU
only)."""
import ctypes

import pytest
import torch

from spion_amd import _lib
from tests.test_gpu_dense_groups import _heads, _module
from tests.test_gpu_split_products import EPS, LIMITS, LOG2E, _bounds, _compare, _special, compare_by_element, improbable

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


def _shared_tiles(mod, tensors):
    """Gradients of a backward without scratch, which the work-groups that share their tiles have to form"""
    grads = [torch.full_like(tensors[0], float("nan")) for _ in range(3)]
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        _call(mod, tensors, grads)
        torch.cuda.synchronize()
    names = " ".join(e.key for e in prof.key_averages())
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert "dense_group_row_kernel<32>" in names and "dense_group_col_kernel<32>" in names, names
        assert "dense_group_col_dq_kernel" not in names
    return grads


# strips a multiple of a group and not (wavefronts without a strip of their own), one tile and one more than a double buffer,
# several groups to a CU
@pytest.mark.parametrize("L,B,H,layout,masked", [(128, 64, 4, "plain", False), (96, 128, 2, "proj", True), (224, 128, 2, "fused", False),
                                                 (1056, 20, 2, "plain", True)])
def test_shared_tiles_match_float64(L, B, H, layout, masked):
    d = 32
    gen = torch.Generator(device="cuda").manual_seed(L + d)
    operands = _heads(B, H, L, d, layout, 3, gen) + _heads(B, H, L, d, "plain", 1, gen)
    mask = torch.ones(B, L, device="cuda")
    if masked:
        mask[0, L // 2:] = 0
        mask[-1, 5:] = 0
    mod, cpp, t = _forward(B, H, L, layout, masked, operands, mask)
    got = _shared_tiles(mod, t)
    cpp.destroy(mod.attn_handle)
    for b in (0, B // 2, B - 1):
        ref = [x[b].double().requires_grad_() for x in t[:3]]
        do = t[5][b].double().contiguous()
        s = ref[0] @ ref[1].transpose(-1, -2).contiguous() * d ** -0.5 - (1e6 * (1 - mask[b].double()) if masked else 0)
        p = torch.softmax(s, -1)
        (p @ ref[2]).backward(do)
        bound = _bounds(*(x.detach().contiguous() for x in ref), do, p.detach(), d ** -0.5)[1:]
        for name, x, y, e in zip(("dQ", "dK", "dV"), got, ref, bound):
            worst = float(((x[b].double() - y.grad).abs() / e.clamp_min(1e-300)).max())
            assert worst <= 1.0, f"{name} of sample {b}: {worst} of the bound"


@pytest.mark.parametrize("which", ["q", "k", "v", "do"])
def test_shared_tiles_infinities_nan_and_the_largest_floats(which):
    """A special element in one head: that head against torch's fp32 steps, the others bit for bit as without it."""
    L, B, H, d = 96, 128, 2, 32
    ones = torch.ones(B, L, device="cuda")

    def run(value):
        one = _special(which, value, H, L, d)
        t = {n: torch.cat([x, x.new_ones(B - 1, H, L, d) * torch.linspace(-1, 1, d)]).cuda() for n, x in one.items()}
        mod, cpp, tensors = _forward(B, H, L, "plain", False, [t[n] for n in ("q", "k", "v", "do")], ones)
        res = [tensors[4], *_shared_tiles(mod, tensors)]
        cpp.destroy(mod.attn_handle)
        return one, res

    _, plain = run(0.0)
    for value in LIMITS:
        one, got = run(value)
        if not 1.0 < abs(value) < float("inf"):  # (beside a finite one the special sample's other elements differ too)
            assert all(torch.equal(x[0, 1], y[0, 1]) for x, y in zip(got, plain))
        assert all(torch.equal(x[1:], y[1:]) for x, y in zip(got, plain))
        Q, K, V, dO = (one[n][0, 0].cuda() for n in ("q", "k", "v", "do"))
        s = (Q * (d ** -0.5 * LOG2E)) @ K.t()
        e = torch.exp2(s - torch.fmax(s, torch.tensor(-10.0 * LOG2E, device="cuda")).amax(-1, keepdim=True))
        P = e / e.sum(-1, keepdim=True)
        O = P @ V
        ds = (dO @ V.t() - (dO * O).sum(-1, keepdim=True)) * P
        want = [O, ds @ K * d ** -0.5, ds.t() @ Q * d ** -0.5, P.t() @ dO]
        _compare([x[0, 0].cpu() for x in got], [x.cpu() for x in want], which, value, L + d)


def test_shared_tiles_near_the_smallest_floats():
    L, B, H, d = 96, 128, 2, 32
    gen = torch.Generator(device="cuda").manual_seed(d)
    q, k, v, do = _heads(B, H, L, d, "plain", 4, gen)
    mod, cpp, t = _forward(B, H, L, "plain", False, (q, k, v, do * 2.0 ** -117), torch.ones(B, L, device="cuda"))
    got = _shared_tiles(mod, t)
    cpp.destroy(mod.attn_handle)
    ref = [x[3].double().requires_grad_() for x in (q, k, v)]
    p = torch.softmax(ref[0] @ ref[1].transpose(-1, -2).contiguous() * d ** -0.5, -1)
    (p @ ref[2]).backward(t[5][3].double())
    for x, y in zip(got, ref):
        assert float((x[3].double() - y.grad).norm() / y.grad.norm()) < 2 * L ** 0.5 * EPS


@pytest.mark.parametrize("L,B", [(96, 128), (1056, 20)])
def test_shared_tiles_and_a_small_row_among_ordinary_ones(L, B):
    H, d = 2, 32
    one = improbable(H, L, d, L + d)
    t = {n: torch.cat([x, torch.randn(B - 1, H, L, d, generator=torch.Generator().manual_seed(1))]).cuda() for n, x in one.items()}
    mod, cpp, tensors = _forward(B, H, L, "plain", False, [t[n] for n in ("q", "k", "v", "do")], torch.ones(B, L, device="cuda"))
    grads = _shared_tiles(mod, tensors)
    cpp.destroy(mod.attn_handle)
    compare_by_element(one, tensors[3][0].transpose(1, 2), tensors[4][0], [x[0] for x in grads], d)
