"""Heads of element patterns launched in groups: the rule (host logic, no device needed), and that every head's results are those
of the same operands elsewhere in the batch, whatever group either lies in (on a GPU only)."""
import pytest
import torch

from spion_amd import _lib
from tests.test_gpu_remainder import _module, _pattern


def _rounds(heads, length, cus):
    """Of work-groups of 256 rows, one per CU; those of 512 rows count 1.6 times."""
    one, two = (-(-heads * -(-length // per) // cus) for per in (256, 512))
    return 1.6 * two if 10 * one > 16 * two else one


@pytest.mark.parametrize("length", [512, 1056, 2048, 4096, 16384])
@pytest.mark.parametrize("unit", [1, 3, 8])
def test_groups_are_whole_units_and_take_no_more_rounds(length, unit):
    for samples in list(range(1, 40)) + [64, 171, 512]:
        for mb in (0.3, 2.0, 4.6, 5.9, 40.0):
            heads, cus = samples * unit, 256
            n = _lib.core().spion_debug_remainder_heads(heads, length, unit, mb * 1e6, cus)
            assert 0 < n <= heads and n % unit == 0
            if heads * mb <= 192.0:
                assert n == heads
            last = heads % n
            assert heads // n * _rounds(n, length, cus) + (_rounds(last, length, cus) if last else 0) <= _rounds(heads, length, cus) + 1e-9


def test_the_sizes_the_rule_was_measured_at():
    pick = lambda heads, mb: _lib.core().spion_debug_remainder_heads(heads, 4096, 2, mb * 1e6, 256)
    assert [pick(h, 4.6) for h in (16, 32, 64, 128)] == [16, 32, 32, 32]
    assert [pick(h, 5.9) for h in (16, 32, 64, 128)] == [16, 32, 32, 32]
    for bad in ((0, 4096, 1), (4, 0, 1), (4, 4096, 0), (5, 4096, 2)):
        assert _lib.core().spion_debug_remainder_heads(*bad, 1e6, 256) == -1


# groups of equal size; a smaller last one; one sample's heads a group; key masks; strided heads
@pytest.mark.gpu
@pytest.mark.parametrize("B,H,L,masked,views", [(320, 2, 1056, False, False), (111, 3, 2048, True, False), (37, 8, 2080, True, True),
                                                (23, 8, 4096, False, True), (136, 2, 2048, False, True)])
def test_heads_do_not_depend_on_their_group(B, H, L, masked, views):
    gen = torch.Generator(device="cuda").manual_seed(L + B)
    pattern = _pattern(L, gen)
    entries = int(pattern.sum())
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:  # P alone makes it more than one group
        assert _lib.core().spion_debug_remainder_heads(B * H, L, H, 4.0 * entries, 256) < B * H
    kinds = 4  # samples of four kinds in no order
    kind = torch.randint(kinds, (B,), generator=gen, device="cuda")
    kind[:kinds], kind[-1] = torch.arange(kinds, device="cuda"), 1

    def operand():
        x = torch.randn(kinds, H, L, 32, generator=gen, device="cuda")[kind]
        return x.transpose(1, 2).contiguous().transpose(1, 2) if views else x

    q, k, v, do = (operand() for _ in range(4))
    valid = torch.ones(kinds, L, device="cuda")
    if masked:
        valid[1, L // 2:] = 0
        valid[3, 100:] = 0
    valid = valid[kind]
    cpp, handle, module = _module(B, H, L, masked)
    leaves = [t.requires_grad_() for t in (q, k, v)]
    out, p = module(*leaves, valid, pattern)
    out.backward(do)
    assert _lib.core().spion_debug_counter(handle, 3) == 1  # by ranges
    assert torch.isfinite(out).all()
    for x in [out.detach(), *(t.grad for t in leaves)] + ([] if masked else [p.detach().view(B, H, -1)]):
        for b in range(B):
            assert torch.equal(x[b], x[int(kind[b])]), b
    cpp.destroy(handle)
