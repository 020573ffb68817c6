"""The fp32 tile kernels' products on the bf16 matrix pipe (operands split into three parts), against float64 with
bounds that scale with the operands (GPU box only)."""
import pytest
import torch

import spion_amd
from oracle import sparse_attention as osa
from spion_amd import workloads

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -24


def _bounds(q, k, v, do, p, scale):
    """Largest errors of O, dQ, dK, dV.  A product of n terms has at most n + 8 roundings of the running sum of
    magnitudes (the splits drop less than one of them per term); a logit's error enters its probability and the
    denominator, the denominator adds one rounding per term of its longest partial sum; a softmax gradient adds its
    two products' errors and its probability's."""
    L, d = q.shape[-2:]
    rnd = lambda n: (n + 8) * EPS
    ab = lambda x, y: x.abs() @ y.abs()
    relp = 2 * rnd(d) * (ab(q, k.transpose(-1, -2)) * scale).amax(-1, keepdim=True) + rnd(L)
    eo = (relp + rnd(L)) * ab(p, v)
    dp, mag = do @ v.transpose(-1, -2), ab(do, v.transpose(-1, -2))
    o = p @ v
    g, gmag = (do * o).sum(-1, keepdim=True), (do.abs() * (o.abs() + eo)).sum(-1, keepdim=True)
    ds = p * (dp - g)
    eds = p * (rnd(d) * (mag + gmag) + (do.abs() * eo).sum(-1, keepdim=True)) + (relp + rnd(2)) * p * (mag + gmag)
    edq = scale * (eds @ k.abs() + rnd(L) * ab(ds, k))
    edk = scale * (eds.transpose(-1, -2) @ q.abs() + rnd(L) * ab(ds.transpose(-1, -2), q))
    edv = (p * relp).transpose(-1, -2) @ do.abs() + rnd(L) * ab(p.transpose(-1, -2), do)
    return eo, edq, edk, edv


# one tile; odd tiles; a strip at and past the registers of four wavefronts (16 and 20 tiles at d = 64, 32 at d = 32); the
# two sweeps (d = 64: most strips beyond 24 tiles; d = 32: beyond 32); heads as views of a projection (row-major tiles)
@pytest.mark.parametrize("d", [32, 64])
@pytest.mark.parametrize("L,extra,strided", [(32, 0.0, False), (96, 1.0, False), (96, 1.0, True), (512, 1.0, False),
                                             (640, 0.9, False), (640, 0.9, True), (1088, 1.0, False)])
def test_wide_ranges_match_float64(d, L, extra, strided):
    B, H, bs = 1, 2, 32
    mat = workloads.band_random_block_mask(L // bs, 1, extra_frac=extra, seed=L + d)
    g = torch.Generator().manual_seed(L * d)
    wide = torch.exp2(torch.randint(-30, 31, (d,), generator=g).float())  # each feature of V and dO has its own scale
    q, k, v, do = (torch.randn(B, H, L, d, generator=g) for _ in range(4))
    v, do = v * wide, do / wide
    cfg = dict(head_dim=d, num_head=H, max_seq_len=L, batch_size=B, block_size=bs)
    cpp = spion_amd.Attention._blockcuda_compile_module()
    handle = cpp.init(d, L, B * H, bs)
    mod = spion_amd.CUDABlockAttention(cfg, cpp, handle)

    def place(t):
        t = t.cuda()
        return (t.transpose(1, 2).contiguous().transpose(1, 2) if strided else t).requires_grad_()

    qc, kc, vc = place(q), place(k), place(v)
    out, _ = mod(qc, kc, vc, torch.ones(B, L, device="cuda"), torch.from_numpy(mat).cuda())
    out.backward(do.cuda())
    pat = torch.from_numpy(mat).double().repeat_interleave(bs, 0).repeat_interleave(bs, 1)
    ref = [t.double().requires_grad_() for t in (q, k, v)]
    o, p = osa.dense_masked_attention(*ref, pat)
    o.backward(do.double())
    bound = _bounds(*(t.detach() for t in ref), do.double(), p.detach(), d ** -0.5)
    got = (out, qc.grad, kc.grad, vc.grad)
    for name, x, y, e in zip(("out", "dQ", "dK", "dV"), got, (o, ref[0].grad, ref[1].grad, ref[2].grad), bound):
        worst = float(((x.detach().double().cpu() - y.detach()).abs() / e).max())
        assert worst <= 1.0, f"{name}: {worst} of the bound"
    cpp.destroy(handle)
