"""The dense backward whose work-groups share their tiles (launches that fill the machine) against float64, and where
elements are infinite, NaN or at the ends of the range (on a GPU only)."""
import pytest
import torch

import spion_amd
from tests.test_gpu_split_products import EPS, LIMITS, LOG2E, _bounds, _compare, _special, compare_by_element, improbable

pytestmark = pytest.mark.gpu


def _heads(B, H, L, d, layout, n, gen):
    """n tensors [B, H, L, d]: plain, or views of a projection's [B, L, H*d] or of a fused one's [B, L, n*H*d]"""
    if layout == "plain":
        return [torch.randn(B, H, L, d, generator=gen, device="cuda") for _ in range(n)]
    if layout == "proj":
        return [torch.randn(B, L, H, d, generator=gen, device="cuda").transpose(1, 2) for _ in range(n)]
    return [t.transpose(1, 2) for t in torch.randn(B, L, n, H, d, generator=gen, device="cuda").unbind(2)]


def _module(B, H, L, d, masked):
    cpp = getattr(spion_amd.Attention, "_cuda_mask_compile_module" if masked else "_cuda_compile_module")()
    cls = spion_amd.CUDAMaskAttention if masked else spion_amd.CUDAAttention
    mod = cls(dict(head_dim=d, num_head=H, max_seq_len=L, batch_size=B), cpp, cpp.init(d, L, B * H))
    assert mod.reads_views
    return mod, cpp


def _step(mod, qkv, do, mask, shared):
    """One step; checks which backward kernels ran."""
    q, k, v = (t.detach().requires_grad_() for t in qkv)
    out, _ = mod(q, k, v, mask)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        out.backward(do)
        torch.cuda.synchronize()
    names = " ".join(e.key for e in prof.key_averages())
    assert ("dense_group_row" in names) == shared and ("dense_group_col" in names) == shared
    assert ("dense_bwd_row" in names) == (not shared) and ("dense_bwd_col" in names) == (not shared)
    return [x.detach() for x in (out, q.grad, k.grad, v.grad)]


# strips a multiple of a group and not (wavefronts without a strip of their own), one tile and one more than a double
# buffer, several groups to a CU; and just below the rule
@pytest.mark.parametrize("d,L,B,H,layout,masked,shared", [
    (32, 128, 64, 4, "plain", False, True), (32, 96, 128, 2, "proj", True, True), (32, 224, 128, 2, "fused", False, True),
    (32, 1056, 20, 2, "plain", True, True), (32, 32, 1024, 1, "plain", False, False), (32, 1024, 10, 1, "proj", False, False),
    (64, 256, 64, 4, "proj", False, True), (64, 160, 128, 2, "plain", True, True), (64, 288, 64, 2, "fused", False, True),
    (64, 1024, 16, 2, "plain", False, True), (64, 1024, 10, 2, "plain", False, False)])
def test_shared_tiles_match_float64(d, L, B, H, layout, masked, shared):
    gen = torch.Generator(device="cuda").manual_seed(L + d)
    q, k, v = _heads(B, H, L, d, layout, 3, gen)
    (do,) = _heads(B, H, L, d, "proj" if layout != "plain" else "plain", 1, gen)
    mask = torch.ones(B, L, device="cuda")
    if masked:
        mask[0, L // 2:] = 0
        mask[-1, 5:] = 0
    mod, cpp = _module(B, H, L, d, masked)
    got = _step(mod, (q, k, v), do, mask, shared)
    cpp.destroy(mod.attn_handle)
    for b in (0, B // 2, B - 1):
        ref = [t[b].double().requires_grad_() for t in (q, k, v)]
        s = ref[0] @ ref[1].transpose(-1, -2).contiguous() * d ** -0.5 - (1e6 * (1 - mask[b].double()) if masked else 0)
        p = torch.softmax(s, -1)
        o = p @ ref[2]
        o.backward(do[b].double())
        bound = _bounds(*(t.detach() for t in ref), do[b].double(), p.detach(), d ** -0.5)
        for name, x, y, e in zip(("out", "dQ", "dK", "dV"), got, (o, *(t.grad for t in ref)), bound):
            # (a masked key's gradients are exact zeros on both sides)
            worst = float(((x[b].double() - y.detach()).abs() / e.clamp_min(1e-300)).max())
            assert worst <= 1.0, f"{name} of sample {b}: {worst} of the bound"


@pytest.mark.parametrize("d,L,B", [(32, 96, 128), (64, 160, 128)])
@pytest.mark.parametrize("which", ["q", "k", "v", "do"])
def test_shared_tiles_infinities_nan_and_the_largest_floats(which, d, L, B):
    """A special element in one head: that head against torch's fp32 steps, the others bit for bit as without it."""
    H = 2
    mod, cpp = _module(B, H, L, d, False)
    mask = torch.ones(B, L, device="cuda")

    def run(value):
        one = _special(which, value, H, L, d)
        t = {n: torch.cat([x, x.new_ones(B - 1, H, L, d) * torch.linspace(-1, 1, d)]).cuda() for n, x in one.items()}
        return one, _step(mod, [t[n] for n in "qkv"], t["do"], mask, True)

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


@pytest.mark.parametrize("d,L,B", [(32, 96, 128), (64, 160, 128)])
def test_shared_tiles_near_the_smallest_floats(d, L, B):
    """As test_gradients_near_the_smallest_floats."""
    H = 2
    gen = torch.Generator(device="cuda").manual_seed(d)
    q, k, v, do = _heads(B, H, L, d, "plain", 4, gen)
    do = do * 2.0 ** -117
    mod, cpp = _module(B, H, L, d, False)
    got = _step(mod, (q, k, v), do, torch.ones(B, L, device="cuda"), True)
    cpp.destroy(mod.attn_handle)
    ref = [t[3].double().requires_grad_() for t in (q, k, v)]
    p = torch.softmax(ref[0] @ ref[1].transpose(-1, -2).contiguous() * d ** -0.5, -1)
    (p @ ref[2]).backward(do[3].double())
    for x, y in zip(got[1:], ref):
        assert float((x[3].double() - y.grad).norm() / y.grad.norm()) < 2 * L ** 0.5 * EPS


# (and the kernels whose wavefronts have tiles of their own, row-major and feature-major)
@pytest.mark.parametrize("d,L,B,views", [(32, 96, 128, True), (32, 1056, 20, True), (64, 160, 128, True), (32, 96, 2, True),
                                         (32, 96, 2, False), (64, 160, 2, True)])
def test_a_small_row_among_ordinary_ones(d, L, B, views):
    H = 2
    one = improbable(H, L, d, L + d)
    t = {n: torch.cat([x, torch.randn(B - 1, H, L, d, generator=torch.Generator().manual_seed(1))]).cuda() for n, x in one.items()}
    mod, cpp = _module(B, H, L, d, False)
    mod.reads_views = views
    leaves = [t[n].requires_grad_() for n in "qkv"]
    out, p = mod(*leaves, torch.ones(B, L, device="cuda"))
    out.backward(t["do"])
    cpp.destroy(mod.attn_handle)
    compare_by_element(one, p.detach()[0], out.detach()[0], [x.grad[0] for x in leaves], d)
