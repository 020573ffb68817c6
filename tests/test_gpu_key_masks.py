"""Key masks that the forward's kernels read themselves, against the penalties 1e6 (1 - mask) made ahead of them: the same bits
for masks of zeros and ones, in every family of kernels (a mask of another type takes the penalties)."""
import numpy as np
import pytest
import torch

import spion_amd
from spion_amd import _lib, workloads
from spion_amd.attention import Attention

pytestmark = pytest.mark.gpu


def _config(B, H, L, d, bs):
    return dict(head_dim=d, num_head=H, max_seq_len=L, batch_size=B, block_size=bs, transformer_dim=H * d, attention_dropout=0.0,
                task="lra-text")


def _element(L, window, per_row):
    sm, off, col = workloads.window_random_csr(L, window, per_row, seed=3)
    mat = np.zeros((L, L), dtype=np.float32)
    mat[np.repeat(np.arange(L), sm), col] = 1.0
    return torch.from_numpy(mat).cuda()


def _heads(B, H, L, d, layout, dtype=torch.float32):
    g = torch.Generator().manual_seed(L + d)
    t = [(torch.randn(B, L, H, d, generator=g) / (8 if dtype == torch.bfloat16 else 1)).to("cuda", dtype).transpose(1, 2) for _ in range(3)]
    return t if layout == "views" else [x.contiguous() for x in t]


def _mask(B, L):
    m = workloads.valid_length_mask(B, L, max(1, L // 3), L, seed=5).cuda()
    if B > 1:
        m[-1] = 0.0  # a sample without a key
    return m


def _same(run, mask):
    partly = torch.where(mask > 0, 1.0 - 1e-6 * torch.arange(mask.shape[1], device="cuda") / 64, 0.0)
    with torch.no_grad():
        here, ref, odd, odd_ref = run(mask), run(mask.double()), run(partly), run(partly.double())
    # the kernels' term fmaf(mask, 1e6, -1e6), or that times log2 e, and the penalty made ahead of them, of L / 64 at most,
    # round two or three times differently: a logit differs by 2^-22 of the penalty, as much of a probability
    part = 2.0 ** -22 * (4 + mask.shape[1] / 64)
    for a, b, c, d in zip(here, ref, odd, odd_ref):
        if not torch.is_tensor(a):  # the key-mask modules return no probabilities
            continue
        assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.isnan(), c.isnan())  # rows without a key, full rows of a pattern
        assert torch.equal(a.nan_to_num(), b.nan_to_num())
        assert torch.equal(c.isnan(), d.isnan()) and (a.isnan().all() or not torch.equal(a.nan_to_num(), c.nan_to_num()))
        c, d = c.nan_to_num().double(), d.nan_to_num().double()
        # a weighted mean of values up to |V|max (probabilities: of ones), each weight and the denominator off by `part`; bf16: one
        # more unit in the last place of the result
        unit = 2.0 ** -7 if a.dtype == torch.bfloat16 else 2.0 ** -22
        assert ((c - d).abs() <= 2 * part * max(1.0, float(d.abs().max())) + unit * d.abs()).all()


# blocks of 32 and 64, strips for one and four wavefronts, two sweeps (every block), ragged numbers of strips, three heads
@pytest.mark.parametrize("layout", ["contiguous", "views"])
@pytest.mark.parametrize("B,H,L,d,bs,extra", [(2, 3, 96, 32, 32, 0.3), (3, 2, 512, 32, 64, 0.1), (2, 2, 1056, 32, 32, 1.0), (64, 2, 1024, 32, 32, 0.05),
                                              (2, 3, 224, 64, 32, 0.3), (2, 1, 1056, 64, 32, 1.0)])
def test_tile_patterns(B, H, L, d, bs, extra, layout):
    cpp = Attention._blockcuda_mask_compile_module()
    mod = spion_amd.CUDABlockMaskAttention(_config(B, H, L, d, bs), cpp, cpp.init(d, L, B * H, bs))
    mat = torch.from_numpy(workloads.band_random_block_mask(L // bs, 1, extra_frac=extra, seed=3).astype(np.float32)).cuda()
    heads = _heads(B, H, L, d, layout)
    _same(lambda m: mod(*heads, m, mat), _mask(B, L))
    off = torch.zeros(B * L + 1, device="cuda")[1:].view(B, L)  # a mask that starts off 16 bytes
    off.copy_(_mask(B, L))
    with torch.no_grad():
        assert torch.equal(mod(*heads, off, mat)[0].nan_to_num(), mod(*heads, _mask(B, L), mat)[0].nan_to_num())
    cpp.destroy(mod.attn_handle)


# the element kernels (head sizes without others), the hybrid ones without and with the remainder by ranges
@pytest.mark.parametrize("layout", ["contiguous", "views"])
@pytest.mark.parametrize("B,H,L,d", [(2, 3, 160, 16), (2, 2, 130, 64), (1, 2, 128, 128), (2, 3, 256, 32), (32, 2, 1056, 32)])
def test_element_patterns(B, H, L, d, layout):
    cpp = Attention._blockcuda_mask_compile_module()
    mod = spion_amd.CUDABlockMaskAttention(_config(B, H, L, d, 1), cpp, cpp.init(d, L, B * H, 1))
    mat = _element(L, 20, 40)
    heads = _heads(B, H, L, d, layout)
    _same(lambda m: mod(*heads, m, mat), _mask(B, L))
    cpp.destroy(mod.attn_handle)


@pytest.mark.parametrize("mean", [False, True])
@pytest.mark.parametrize("B,H,L,d", [(2, 3, 96, 32), (2, 2, 1024, 32), (1, 3, 1056, 32), (1, 2, 2080, 32), (2, 3, 96, 64), (1, 2, 1056, 64)])
def test_dense(B, H, L, d, mean):
    cpp = Attention._cuda_mask_compile_module()
    mod = spion_amd.CUDAMaskAttention(_config(B, H, L, d, 32), cpp, cpp.init(d, L, B * H))
    mod.emit_score_map = mean
    heads = _heads(B, H, L, d, "views")
    _same(lambda m: (*mod(*heads, m), mod.score_map if mean else None), _mask(B, L))
    cpp.destroy(mod.attn_handle)


# paired strips and single ones, chunks of long strips (a global row), three heads a sample
@pytest.mark.parametrize("layout", ["contiguous", "views"])
@pytest.mark.parametrize("B,H,L,d,bs", [(2, 3, 192, 32, 64), (2, 3, 224, 64, 32), (4, 2, 4096, 64, 64)])
def test_bf16(B, H, L, d, bs, layout):
    mod = spion_amd.BlockAttentionBF16(_config(B, H, L, d, bs), key_mask=True)
    mat_np = workloads.band_random_block_mask(L // bs, 1, extra_frac=0.1, seed=3).astype(np.float32)
    mat_np[0, :] = 1.0
    mat = torch.from_numpy(mat_np).cuda()
    heads = _heads(B, H, L, d, layout, torch.bfloat16)
    _same(lambda m: mod(*heads, m, mat)[:1], _mask(B, L))


def test_refusals():
    core = _lib.core()
    B, H, L, d, bs = 2, 2, 64, 32, 32
    cpp = Attention._blockcuda_mask_compile_module()
    mod = spion_amd.CUDABlockMaskAttention(_config(B, H, L, d, bs), cpp, cpp.init(d, L, B * H, bs))
    idx = mod.csr_cache.get(torch.eye(L // bs, device="cuda"), bs)
    q, k, v = _heads(B, H, L, d, "contiguous")
    mask, out, p = torch.ones(B, L, device="cuda"), torch.empty_like(q), torch.empty(B * H * idx.nnz, device="cuda")
    for m, heads in ((None, H), (mask.data_ptr(), 0), (mask.data_ptr(), 3), (mask.data_ptr() + 4, H)):
        core.spion_attn_forward_rowmajor_keys(mod.attn_handle, q.data_ptr(), k.data_ptr(), v.data_ptr(), m, heads, p.data_ptr(),
                                              out.data_ptr(), *idx.tail)
        assert core.spion_error_pending()
        core.spion_clear_error()
    cpp.destroy(mod.attn_handle)
