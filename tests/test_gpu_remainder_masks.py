"""Element patterns whose heads are launched in groups: key masks that several samples of strided heads share (on a GPU only)."""
import ctypes

import pytest
import torch

from spion_amd import _lib
from spion_amd.csr import block_mask_to_csr_host
from tests.abi_utils import SparseABI
from tests.test_gpu_remainder import _pattern

pytestmark = pytest.mark.gpu


def test_a_mask_row_for_more_heads_than_a_sample_has():
    """Each mask row serves 16 heads, eight samples of the layout: groups of heads begin where both do."""
    B, H, L, shared, core = 136, 2, 2048, 16, _lib.core()
    gen = torch.Generator(device="cuda").manual_seed(3)
    abi = SparseABI(32, L, B * H, 1, with_mask=True)
    abi.set_pattern(*block_mask_to_csr_host(_pattern(L, gen).cpu().numpy(), 1))
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:  # groups of whole samples would begin inside a mask row
        per = core.spion_debug_remainder_heads(B * H, L, H, 4.0 * abi.nnz, 256)
        assert per < B * H and per % shared
    q, k, v = (torch.randn(B, L, H, 32, generator=gen, device="cuda").transpose(1, 2) for _ in range(3))
    keys = torch.randint(L // 4, L + 1, (B * H // shared, 1), generator=gen, device="cuda")
    mask = (torch.arange(L, device="cuda")[None] < keys).float()
    layout = _lib.head_layout(q)
    lay = ctypes.addressof(layout)
    scratch = torch.empty(core.spion_attn_scratch(abi.handle, abi.offsets.data_ptr(), abi.columns.data_ptr(), abi.nnz, 0), device="cuda")

    def forward(mask, heads):
        out, p = torch.full_like(q, float("nan")), torch.full((B * H * abi.nnz,), float("nan"), device="cuda")
        core.spion_attn_forward_scratch(abi.handle, q.data_ptr(), k.data_ptr(), v.data_ptr(), mask.data_ptr(), heads, p.data_ptr(),
                                        out.data_ptr(), abi.offsets.data_ptr(), abi.columns.data_ptr(), abi.nnz, H, lay, lay,
                                        scratch.data_ptr(), scratch.numel())
        _lib.check_error("forward")
        return out, p

    got = forward(mask, shared)
    assert core.spion_debug_counter(abi.handle, 3) == 1  # by ranges
    want = forward(mask.repeat_interleave(shared // H, 0).contiguous(), H)
    abi.close()
    for x, y in zip(got, want):
        assert torch.equal(x.isnan(), y.isnan()) and torch.equal(x.nan_to_num(), y.nan_to_num())
