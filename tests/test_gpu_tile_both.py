"""Both passes of a small backward in one launch (d = 32, patterns of aligned tiles) against float64 and against one pass after
the other (on a GPU only)."""
import pytest
import torch

import spion_amd
from oracle import sparse_attention as osa
from spion_amd import _lib, workloads
from tests.abi_utils import SparseABI
from tests.test_gpu_split_products import EPS, _bounds, _csr

pytestmark = pytest.mark.gpu


def _pattern(L, bs, kind):
    nb = L // bs
    if kind == "full":
        return torch.ones(nb, nb).numpy()
    mat = workloads.band_random_block_mask(nb, 1, density=0.25 if kind == "dense" else 0.136, seed=L)
    if kind == "columns":  # an eighth of the columns full (more than count as long ones); rows and columns with nothing
        mat[:, 2::7] = 1
        mat[3] = 0
        mat[:, 5] = 0
    return mat


def _kernels(fn):
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        fn()
        torch.cuda.synchronize()
    return " ".join(e.key for e in prof.key_averages())


# one tile; a wavefront without tiles; one, two and four wavefronts a strip; empty strips beside long ones; 64x64 blocks; the
# most tiles one launch takes on 256 CUs, and one head more
@pytest.mark.parametrize("strided", [False, True])
@pytest.mark.parametrize("B,H,L,bs,kind,W", [
    (1, 1, 32, 32, "full", 2), (3, 1, 96, 32, "full", 4), (1, 2, 1024, 32, "band", 4), (8, 2, 1024, 32, "band", 2),
    (64, 2, 512, 32, "dense", 1), (5, 3, 672, 32, "columns", 4), (3, 4, 1984, 64, "band", 2), (5, 4, 1024, 32, "full", 1),
    (7, 3, 1024, 32, "full", 0)])
def test_both_passes_match_float64(B, H, L, bs, kind, W, strided):
    d = 32
    mat = _pattern(L, bs, kind)
    gen = torch.Generator(device="cuda").manual_seed(L + B)

    def heads(n):
        shape = (B, L, H, d) if strided else (B, H, L, d)
        t = [torch.randn(*shape, device="cuda", generator=gen) for _ in range(n)]
        return [x.transpose(1, 2) for x in t] if strided else t

    q, k, v, do = heads(4)
    cfg = dict(head_dim=d, num_head=H, max_seq_len=L, batch_size=B, block_size=bs)
    cpp = spion_amd.Attention._blockcuda_compile_module()
    handle = cpp.init(d, L, B * H, bs)
    mod = spion_amd.CUDABlockAttention(cfg, cpp, handle)
    leaves = [t.detach().requires_grad_() for t in (q, k, v)]
    out, _ = mod(*leaves, torch.ones(B, L, device="cuda"), torch.from_numpy(mat).cuda())
    names = _kernels(lambda: out.backward(do))
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert (f"tile_bwd_both_kernel<{W}, " if W else "tile_bwd_col_kernel<32, ") in names, names
        assert ("tile_bwd_row_kernel" in names) == (W == 0)
    cpp.destroy(handle)
    pat = torch.from_numpy(mat).cuda().double().repeat_interleave(bs, 0).repeat_interleave(bs, 1)
    for b in sorted({0, B // 2, B - 1}):
        ref = [t[b].detach().double().contiguous().requires_grad_() for t in (q, k, v)]
        o, p = osa.dense_masked_attention(*ref, pat)
        o.backward(do[b].double())
        bound = _bounds(*(t.detach() for t in ref), do[b].double().contiguous(), p.detach(), d ** -0.5)
        got = (out.detach(), *(t.grad for t in leaves))
        for name, x, y, e in zip(("out", "dQ", "dK", "dV"), got, (o, *(t.grad for t in ref)), bound):
            worst = float(((x[b].double() - y.detach()).abs() / e.clamp_min(1e-300)).max())
            assert worst <= 1.0, f"{name} of sample {b}: {worst} of the bound"


def test_a_gradient_over_an_operand_runs_one_pass_after_the_other():
    core, NB, L, d, bs = _lib.core(), 6, 512, 32, 32
    abi = SparseABI(d, L, NB, bs, False)
    abi.set_pattern(*_csr(workloads.band_random_block_mask(L // bs, 1, density=0.25, seed=1), bs))
    gen = torch.Generator(device="cuda").manual_seed(0)
    q, k, v, do = (torch.randn(NB, L, d, device="cuda", generator=gen) for _ in range(4))
    out, p = abi.forward_rowmajor(q, k, v)

    def backward(over):
        at = {"out": out.clone(), "k": k.clone(), "v": v.clone()}
        grads = [at[over[n]] if n in over else torch.empty_like(q) for n in ("dq", "dk", "dv")]
        ptr = [t.data_ptr() for t in (q, at["k"], at["v"], p, at["out"], do)]
        names = _kernels(lambda: core.spion_attn_backward_rowmajor(
            abi.handle, *ptr, None, *(t.data_ptr() for t in grads), abi.offsets.data_ptr(), abi.columns.data_ptr(),
            abi.sum_mat.data_ptr(), abi.nnz))
        _lib.check_error("backward")
        return names, grads

    names, plain = backward({})
    assert "tile_bwd_both_kernel" in names
    for over in ({"dq": "out"}, {"dk": "out"}, {"dv": "out"}, {"dk": "k"}, {"dv": "k"}, {"dk": "v"}, {"dv": "v"}):
        names, got = backward(over)
        assert "tile_bwd_row_kernel" in names and "tile_bwd_both_kernel" not in names
        for x, y in zip(got, plain):  # sums of at most L + d + 3 roundings each in another order
            assert float((x - y).norm()) <= 2 * (L + d + 3) * EPS * float(y.norm())
    abi.close()
