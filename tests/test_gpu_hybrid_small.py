"""The dense tiles of element patterns, backward, at the low end of the range: their products run on split operands, and sums that
are too small for those on whole ones (on a GPU only)."""
import numpy as np
import pytest
import torch

import spion_amd
from oracle import sparse_attention as osa
from spion_amd import _lib
from tests.test_gpu_split_products import EPS, NAMES, _run_sparse, _special, compare_by_element, improbable

pytestmark = pytest.mark.gpu
L, H, D = 544, 2, 32


def _pattern(half):
    """A window and random columns.  24 to either side: up to three tiles a strip, one wavefront each; 224: fifteen, four."""
    i, g = np.arange(L), np.random.default_rng(half)
    return ((g.random((L, L)) < 20 / L) | (abs(i[:, None] - i[None, :]) <= half)).astype(np.float32)


@pytest.mark.parametrize("half", [24, 224])
@pytest.mark.parametrize("route", ["module", "strided"])
@pytest.mark.parametrize("power", [-100, -112, -117])
def test_gradients_near_the_smallest_floats(power, route, half):
    """As for the tile patterns: at most L roundings of 2^-24 that add up like a random walk, with a margin of two."""
    mat = _pattern(half)
    t = _special("do", 0.0, H, L, D)
    t["do"] = t["do"] * 2.0 ** power
    got, path = _run_sparse(t, mat, 1, False, route)
    assert path == 3
    ref = [t[n].double().requires_grad_() for n in "qkv"]
    osa.dense_masked_attention(*ref, torch.from_numpy(mat).double())[0].backward(t["do"].double())
    for name, x, y in zip(NAMES[1:], got[1:], ref):
        err = float((x.double() - y.grad).norm() / y.grad.norm())
        assert err < 2 * L ** 0.5 * EPS, (name, err)


@pytest.mark.parametrize("half", [24, 224])
@pytest.mark.parametrize("strided", [False, True])
def test_a_small_row_among_ordinary_ones(strided, half):
    t, mat = improbable(H, L, D, L + D), _pattern(half)
    cpp = spion_amd.Attention._blockcuda_compile_module()
    handle = cpp.init(D, L, H, 1)
    mod = spion_amd.CUDABlockAttention(dict(head_dim=D, num_head=H, max_seq_len=L, batch_size=1, block_size=1), cpp, handle)
    place = lambda x: x.cuda().transpose(1, 2).contiguous().transpose(1, 2) if strided else x.cuda()
    leaves = [place(t[n]).requires_grad_() for n in "qkv"]
    out, p = mod(*leaves, torch.ones(1, L, device="cuda"), torch.from_numpy(mat).cuda())
    out.backward(t["do"].cuda())
    assert _lib.core().spion_last_path(handle) == 3
    full = torch.zeros(H, L, L, device="cuda")
    full[:, torch.from_numpy(mat).cuda() > 0] = p.detach().reshape(H, -1)
    compare_by_element(t, full, out.detach()[0], [x.grad[0] for x in leaves], D)
    cpp.destroy(handle)
