"""The remainder kernels that hold their gathered operands in LDS, at lengths that are no multiple of their work-groups or
ranges (rows, columns and keys past the end), against float64 on some of the heads (on a GPU only)."""
import pytest
import torch

import spion_amd
from spion_amd import _lib

pytestmark = pytest.mark.gpu


def _reference(q, k, v, do, pattern, valid):
    q, k, v = (t.double().requires_grad_() for t in (q, k, v))
    s = q @ k.transpose(-1, -2).contiguous() / q.shape[-1] ** 0.5
    if valid is not None:
        s = s - 1e6 * (1.0 - valid.double())[:, None, :]
    p = torch.softmax(s * pattern, -1) * pattern
    o = p @ v
    o.backward(do.double())
    return o.detach(), q.grad, k.grad, v.grad


# column pass with two, four and eight columns per lane group; logits and P.V from LDS where they fill the machine; no dense
# structure ("uniform": the element kernels, whose column pass is the same kernel)
@pytest.mark.parametrize("B,H,L,kind,masked", [(17, 3, 1056, "window", False), (17, 5, 1504, "window", True),
                                               (64, 2, 2016, "window", False), (64, 2, 2016, "window", True),
                                               (17, 5, 1504, "uniform", False)])
def test_ragged_lengths(B, H, L, kind, masked):
    d, dev = 32, "cuda"
    gen = torch.Generator(device=dev).manual_seed(L + B)
    i = torch.arange(L, device=dev)
    pattern = (torch.rand(L, L, generator=gen, device=dev) < (35 / L if kind == "window" else 0.05)).float()
    if kind == "window":
        pattern[(i[:, None] - i[None, :]).abs() <= 24] = 1.0
    pattern[5] = 0.0
    pattern[:, L - 2] = 0.0
    pattern[L - 1, L - 1] = 1.0
    q, k, v = (torch.randn(B, H, L, d, generator=gen, device=dev).requires_grad_() for _ in range(3))
    do = torch.randn(B, H, L, d, generator=gen, device=dev)
    valid = torch.ones(B, L, device=dev)
    if masked:
        valid = (i[None, :] < torch.randint(L // 2, L + 1, (B, 1), generator=gen, device=dev)).float()
    cfg = dict(head_dim=d, num_head=H, max_seq_len=L, batch_size=B, block_size=1)
    load, cls = (("_blockcuda_mask_compile_module", spion_amd.CUDABlockMaskAttention) if masked else
                 ("_blockcuda_compile_module", spion_amd.CUDABlockAttention))
    cpp = getattr(spion_amd.Attention, load)()
    handle = cpp.init(d, L, B * H, 1)
    out, _ = cls(cfg, cpp, handle)(q, k, v, valid, pattern)
    out.backward(do)
    torch.cuda.synchronize()
    assert _lib.core().spion_last_path(handle) == (3 if kind == "window" else 2)
    for b, h in ((0, 0), (B // 2, H - 1), (B - 1, H - 1)):
        at = lambda t: t.detach()[b, h][None]
        ref = _reference(at(q), at(k), at(v), at(do), pattern.double()[None], valid[b][None] if masked else None)
        for name, x, y in zip(("out", "dQ", "dK", "dV"), (out, q.grad, k.grad, v.grad), ref):
            # a few hundred terms each: 2^-24 of a typical element per rounding, with a wide margin
            tol = 2e-5 * (y.abs() + y.pow(2).mean().sqrt())
            worst = float(((at(x).double() - y).abs() / tol).max())
            assert worst <= 1.0, f"{name}, head {(b, h)}: {worst}"
    cpp.destroy(handle)
