"""Element patterns whose heads are launched in groups: gradients over operands of heads still to come (on a GPU only)."""
import ctypes

import pytest
import torch

from spion_amd import _lib
from spion_amd.csr import block_mask_to_csr_host
from tests.abi_utils import SparseABI
from tests.test_gpu_remainder import _pattern

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("views", [False, True])
def test_a_gradient_over_operands_of_other_heads_keeps_all_heads_together(views):
    """dK of a sample lies over K of the one before: the column launches of all heads come behind the row launches, which alone
    read K.  In groups, the last first, K of the earlier heads would be gone."""
    B, H, L, core = 136, 2, 2048, _lib.core()
    gen = torch.Generator(device="cuda").manual_seed(4)
    abi = SparseABI(32, L, B * H, 1, with_mask=False)
    abi.set_pattern(*block_mask_to_csr_host(_pattern(L, gen).cpu().numpy(), 1))

    def heads(n, make=lambda *s: torch.randn(*s, generator=gen, device="cuda")):
        return make(n, L, H, 32).transpose(1, 2) if views else make(n, H, L, 32)

    q, v, do, out = (heads(B) for _ in range(4))
    kbuf = heads(B + 1)
    k, p = kbuf[1:], torch.empty(B * H * abi.nnz, device="cuda")
    layout = _lib.head_layout(q)
    lay = (ctypes.addressof(layout),) if views else (None,)
    index = [abi.offsets.data_ptr(), abi.columns.data_ptr()]
    scratch = torch.empty(max(core.spion_attn_scratch(abi.handle, *index, abi.nnz, b) for b in (0, 1)), device="cuda")
    tail = (scratch.data_ptr(), scratch.numel())
    core.spion_attn_forward_scratch(abi.handle, q.data_ptr(), k.data_ptr(), v.data_ptr(), None, 0, p.data_ptr(), out.data_ptr(),
                                    *index, abi.nnz, H, *lay * 2, *tail)
    _lib.check_error("forward")
    assert core.spion_debug_counter(abi.handle, 3) == 1  # by ranges

    def backward(k, dk):
        grads = [heads(B, lambda *s: torch.empty(*s, device="cuda")) if g is None else g for g in (None, dk, None)]
        ptr = [t.data_ptr() for t in (q, k, v, p, out, do, *grads)]
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
            core.spion_attn_backward_scratch(abi.handle, *ptr, *index, abi.nnz, H, *lay * 3, *tail)
            torch.cuda.synchronize()
        _lib.check_error("backward")
        return sum(e.count for e in prof.key_averages() if "hyb_tile_bwd_row" in e.key), grads

    groups, want = backward(k, None)
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert groups > 1
    groups, got = backward(k, kbuf[:-1])
    assert groups == 1
    abi.close()
    for x, y in zip(got, want):  # sums of at most L + 35 roundings each in another order
        assert float((x - y).norm()) <= 2 * (L + 35) * 2.0 ** -24 * float(y.norm())
