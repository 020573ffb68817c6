"""The dense backward in one walk over the map (head dimension 32, launches that fill most of the machine) against float64, where
elements are infinite, NaN or at the ends of the range, and without scratch (on a GPU only)."""
import ctypes

import pytest
import torch

from spion_amd import _lib
from tests.test_gpu_dense_groups import _heads, _module
from tests.test_gpu_split_products import EPS, LIMITS, LOG2E, _bounds, _compare, _special, compare_by_element, improbable

pytestmark = pytest.mark.gpu


def _step(mod, qkv, do, mask, G):
    """One step; checks that G strips went to a work-group."""
    q, k, v = (t.detach().requires_grad_() for t in qkv)
    out, _ = mod(q, k, v, mask)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        out.backward(do)
        torch.cuda.synchronize()
    names = " ".join(e.key for e in prof.key_averages())
    assert f"dense_group_col_dq_kernel<{G}>" in names and "dense_group_row_sum" in names
    return [x.detach() for x in (out, q.grad, k.grad, v.grad)]


# two tiles; a last group of one strip and of all but one; one part and several; groups of four and eight; more than one round
@pytest.mark.parametrize("L,B,H,layout,masked,G", [
    (64, 256, 1, "plain", False, 4), (96, 64, 3, "fused", True, 4), (160, 128, 4, "proj", False, 4), (288, 50, 2, "plain", True, 8),
    (224, 128, 2, "fused", False, 8), (320, 32, 4, "proj", True, 8), (1056, 20, 2, "plain", True, 8), (2048, 12, 1, "proj", False, 4),
    (1024, 128, 1, "fused", False, 8)])
def test_one_walk_matches_float64(L, B, H, layout, masked, G):
    d = 32
    gen = torch.Generator(device="cuda").manual_seed(L + B)
    q, k, v = _heads(B, H, L, d, layout, 3, gen)
    (do,) = _heads(B, H, L, d, "proj" if layout != "plain" else "plain", 1, gen)
    mask = torch.ones(B, L, device="cuda")
    if masked:
        mask[0, L // 2:] = 0
        mask[-1, 5:] = 0
    mod, cpp = _module(B, H, L, d, masked)
    got = _step(mod, (q, k, v), do, mask, G)
    cpp.destroy(mod.attn_handle)
    for b in (0, B // 2, B - 1):
        ref = [t[b].double().requires_grad_() for t in (q, k, v)]
        s = ref[0] @ ref[1].transpose(-1, -2).contiguous() * d ** -0.5 - (1e6 * (1 - mask[b].double()) if masked else 0)
        p = torch.softmax(s, -1)
        o = p @ ref[2]
        o.backward(do[b].double())
        bound = _bounds(*(t.detach() for t in ref), do[b].double(), p.detach(), d ** -0.5)
        for name, x, y, e in zip(("out", "dQ", "dK", "dV"), got, (o, *(t.grad for t in ref)), bound):
            worst = float(((x[b].double() - y.detach()).abs() / e.clamp_min(1e-300)).max())
            assert worst <= 1.0, f"{name} of sample {b}: {worst} of the bound"


@pytest.mark.parametrize("which", ["q", "k", "v", "do"])
def test_one_walk_infinities_nan_and_the_largest_floats(which):
    """A special element in one head: that head against torch's fp32 steps, the others bit for bit as without it."""
    L, B, H, d, G = 288, 50, 2, 32, 8
    mod, cpp = _module(B, H, L, d, False)
    mask = torch.ones(B, L, device="cuda")

    def run(value):
        one = _special(which, value, H, L, d)
        t = {n: torch.cat([x, x.new_ones(B - 1, H, L, d) * torch.linspace(-1, 1, d)]).cuda() for n, x in one.items()}
        return one, _step(mod, [t[n] for n in "qkv"], t["do"], mask, G)

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
    cpp.destroy(mod.attn_handle)


def test_one_walk_near_the_smallest_floats_and_a_small_row():
    L, B, H, d, G = 288, 50, 2, 32, 8
    gen = torch.Generator(device="cuda").manual_seed(d)
    mod, cpp = _module(B, H, L, d, False)
    mask = torch.ones(B, L, device="cuda")
    q, k, v, do = _heads(B, H, L, d, "plain", 4, gen)
    do = do * 2.0 ** -117
    got = _step(mod, (q, k, v), do, mask, G)
    ref = [t[3].double().requires_grad_() for t in (q, k, v)]
    p = torch.softmax(ref[0] @ ref[1].transpose(-1, -2).contiguous() * d ** -0.5, -1)
    (p @ ref[2]).backward(do[3].double())
    for x, y in zip(got[1:], ref):
        assert float((x[3].double() - y.grad).norm() / y.grad.norm()) < 2 * L ** 0.5 * EPS
    one = improbable(H, L, d, L + d)
    t = {n: torch.cat([x, torch.randn(B - 1, H, L, d, generator=torch.Generator().manual_seed(1))]).cuda() for n, x in one.items()}
    leaves = [t[n].requires_grad_() for n in "qkv"]
    out, p = mod(*leaves, mask)
    out.backward(t["do"])
    cpp.destroy(mod.attn_handle)
    compare_by_element(one, p.detach()[0], out.detach()[0], [x.grad[0] for x in leaves], d)


def test_calls_without_enough_scratch_or_over_an_operand_run_the_two_passes():
    core, NB, L, d = _lib.core(), 100, 288, 32
    gen = torch.Generator(device="cuda").manual_seed(0)
    q, k, v, do = _heads(NB, 1, L, d, "plain", 4, gen)
    h = core.spion_dense_init(d, L, NB)
    core.spion_set_stream(h, torch.cuda.current_stream().cuda_stream)
    layout = _lib.head_layout(q)
    lay = ctypes.addressof(layout)
    attn, out = torch.empty(NB, L, L, device="cuda"), torch.empty_like(q)
    core.spion_dense_forward_strided(h, q.data_ptr(), k.data_ptr(), v.data_ptr(), None, attn.data_ptr(), out.data_ptr(), 1, lay, lay)
    floats = core.spion_dense_scratch(h)
    assert floats == 2 * NB * L * d
    scratch = torch.empty(floats, device="cuda")

    def backward(*tail, dk=None, dv=None):  # (which operand the gradient lies over)
        at = {"k": k.clone(), "v": v.clone(), "out": out.clone()}
        grads = [torch.empty_like(q), at.get(dk, torch.empty_like(q)), at.get(dv, torch.empty_like(q))]
        call = core.spion_dense_backward_scratch if tail else core.spion_dense_backward_strided
        call(h, q.data_ptr(), at["k"].data_ptr(), at["v"].data_ptr(), attn.data_ptr(), at["out"].data_ptr(), do.data_ptr(),
             *(g.data_ptr() for g in grads), 1, lay, lay, lay, *tail)
        _lib.check_error()
        torch.cuda.synchronize()
        return grads

    passes = backward()
    for tail in ((None, 0), (scratch.data_ptr(), floats - 1), (scratch.data_ptr() + 4, floats)):
        assert all(torch.equal(x, y) for x, y in zip(backward(*tail), passes))
    for over in ({"dk": "k"}, {"dk": "v"}, {"dk": "out"}, {"dv": "k"}, {"dv": "v"}, {"dv": "out"}):
        assert all(torch.equal(x, y) for x, y in zip(backward(scratch.data_ptr(), floats, **over), passes))
    walk = backward(scratch.data_ptr(), floats)
    assert not torch.equal(walk[0], passes[0])  # (dQ is summed in another order)
    for x, y in zip(walk, passes):
        assert float((x - y).norm() / y.norm()) < 2 * L ** 0.5 * EPS
    core.spion_dense_destroy(h)
