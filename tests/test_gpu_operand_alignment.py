"""Row-major operands that start off 16 bytes, which kernels that load them into LDS 16 bytes a lane leave to others (on a GPU
only)."""
import numpy as np
import pytest
import torch

from spion_amd import _lib, workloads
from tests.abi_utils import SparseABI
from tests.test_gpu_split_products import EPS, _csr

pytestmark = pytest.mark.gpu


def _off(x):
    """x, four bytes behind a multiple of 16"""
    buf = torch.zeros(x.numel() + 4, device="cuda")
    y = buf[1:x.numel() + 1].view(x.shape)
    y.copy_(x)
    assert y.data_ptr() % 16 == 4
    return y


def _kernels(fn):
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        fn()
        torch.cuda.synchronize()
    return " ".join(e.key for e in prof.key_averages())


def _backward(abi, t):
    """Kernel names and gradients of a row-major backward on {q, k, v, p, out, do}"""
    grads, ds = [torch.empty_like(t["q"]) for _ in range(3)], torch.empty(abi.NB * abi.nnz, device="cuda")
    ptr = [t[n].data_ptr() for n in ("q", "k", "v", "p", "out", "do")]
    names = _kernels(lambda: _lib.core().spion_attn_backward_rowmajor(
        abi.handle, *ptr, ds.data_ptr(), *(x.data_ptr() for x in grads), abi.offsets.data_ptr(), abi.columns.data_ptr(),
        abi.sum_mat.data_ptr(), abi.nnz))
    _lib.check_error("backward")
    return names, grads


def _step(L, NB, mat, bs):
    abi = SparseABI(32, L, NB, bs, False)
    abi.set_pattern(*_csr(mat, bs))
    gen = torch.Generator(device="cuda").manual_seed(L)
    t = {n: torch.randn(NB, L, 32, device="cuda", generator=gen) for n in ("q", "k", "v", "do")}
    t["out"], t["p"] = abi.forward_rowmajor(t["q"], t["k"], t["v"])
    return abi, t


def _close(got, want, L):
    for x, y in zip(got, want):  # sums of at most L + 32 + 3 roundings each in another order
        assert float((x - y).norm()) <= 2 * (L + 35) * EPS * float(y.norm())


@pytest.mark.parametrize("which", ["q", "k", "v", "do"])
def test_tiles_of_element_patterns(which):
    """A pattern whose remainder is gathered: the element kernels."""
    L, i, g = 1056, np.arange(1056), np.random.default_rng(1)
    abi, t = _step(L, 2, ((g.random((L, L)) < 35 / L) | (abs(i[:, None] - i[None, :]) <= 24)).astype(np.float32), 1)
    assert abi.last_path() == 3 and _lib.core().spion_debug_counter(abi.handle, 3) == 0
    names, want = _backward(abi, t)
    assert "hyb_tile_bwd" in names
    names, got = _backward(abi, {**t, which: _off(t[which])})
    assert "hyb_tile_bwd" not in names
    _close(got, want, L)
    abi.close()


def test_output_of_a_small_tile_pattern():
    """Out enters the one launch of both passes as tiles, the two launches row by row."""
    L, bs = 512, 32
    abi, t = _step(L, 6, workloads.band_random_block_mask(L // bs, 1, density=0.25, seed=1), bs)
    names, want = _backward(abi, t)
    assert "tile_bwd_both_kernel" in names and _lib.core().spion_debug_counter(abi.handle, 4) == 1
    names, got = _backward(abi, {**t, "out": _off(t["out"])})
    assert "tile_bwd_row_kernel" in names and "tile_bwd_both_kernel" not in names
    assert _lib.core().spion_debug_counter(abi.handle, 4) == 0
    _close(got, want, L)
    abi.close()
