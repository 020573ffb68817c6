"""The fp32 tile kernels' products on the bf16 matrix pipe (operands split into three parts), against float64 with
bounds that scale with the operands (on a GPU only)."""
import numpy as np
import pytest
import torch

import spion_amd
from oracle import sparse_attention as osa
from spion_amd import _lib, workloads
from tests.abi_utils import SparseABI

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -24
LOG2E = 1.4426950408889634


def _bounds(q, k, v, do, p, scale):
    """Largest errors of O, dQ, dK, dV.  A product of n terms has at most n + 8 roundings of the running sum of
    magnitudes (the splits drop at most about one per term, 2^-24 of it, while the matrix instructions round once in
    sixteen terms); a logit's error enters its probability and the
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


# ---- infinities, NaN and the ends of the range ---------------------------------------------------
LIMITS = [float("inf"), -float("inf"), float("nan"), 2.0 ** 128 - 2.0 ** 104, -(2.0 ** 128 - 2.0 ** 119)]
NAMES = ("out", "dQ", "dK", "dV")


def _special(which, value, H, L, d):
    """Normal operands [1, H, L, d] with one special element in row L/2 + 1 of the first head; feature 3 of K and V is positive,
    so that an infinite q there gives logits of one sign, and probabilities of zero for the negative one.  Beside a
    finite one everything is a sixteenth, so that no product with it overflows, in whatever order it is scaled."""
    g = torch.Generator().manual_seed(L + d)
    t = dict(zip(("q", "k", "v", "do"), (torch.randn(1, H, L, d, generator=g) for _ in range(4))))
    for n in ("k", "v"):
        t[n][..., 3] = t[n][..., 3].abs()
    if 1.0 < abs(value) < float("inf"):
        t = {n: x / 16 for n, x in t.items()}
    t[which][0, 0, L // 2 + 1, 3] = value
    return t


def _kinds(x):
    """0 finite, 1 +inf, 2 -inf, 3 NaN"""
    return torch.isposinf(x) + 2 * torch.isneginf(x) + 3 * torch.isnan(x)


def _compare(got, want, which, value, terms, outputs=4):
    """The same elements infinite and NaN; finite ones agree to the roundings of sums of so many terms of their tensor's
    largest size.  (A finite logit of 2^120 makes its row one-hot: the gradients are rounding noise times 2^128.)"""
    n = 1 if which in ("q", "k") and abs(value) < float("inf") else outputs
    for name, x, y in zip(NAMES[:n], got, want):
        assert torch.equal(_kinds(x), _kinds(y)), (value, name, int((_kinds(x) != _kinds(y)).sum()))
        x, y = (torch.nan_to_num(z.double(), nan=0.0, posinf=0.0, neginf=0.0) for z in (x, y))
        assert float((x - y).abs().max()) <= 16 * terms * EPS * float(y.abs().max()), (value, name)


def _run_sparse(t, mat, bs, element, route):
    _, H, L, d = t["q"].shape
    if route == "abi":  # feature-major K and V, key penalties
        abi = SparseABI(d, L, H, bs, with_mask=True)
        abi.set_pattern(*_csr(mat, bs))
        abi.force_element(element)
        pen = torch.zeros(H, L, device="cuda")
        pen[:, L // 3] = 1e6
        q, k, v, do = (t[n][0].cuda() for n in ("q", "k", "v", "do"))
        O, P = abi.forward(q, k, v, pen)
        res, path = [O, *abi.backward(q, k, v, P, do)], abi.last_path()
        abi.close()
        return [x.cpu() for x in res], path
    cfg = dict(head_dim=d, num_head=H, max_seq_len=L, batch_size=1, block_size=bs)
    cpp = spion_amd.Attention._blockcuda_compile_module()
    handle = cpp.init(d, L, H, bs)
    _lib.core().spion_force_element_path(handle, int(element))
    mod = spion_amd.CUDABlockAttention(cfg, cpp, handle)
    place = lambda x: x.cuda().transpose(1, 2).contiguous().transpose(1, 2) if route == "strided" else x.cuda()
    q, k, v = (place(t[n]).requires_grad_() for n in "qkv")
    out, _ = mod(q, k, v, torch.ones(1, L, device="cuda"), torch.from_numpy(mat).cuda())
    out.backward(t["do"].cuda())
    path = _lib.core().spion_last_path(handle)
    cpp.destroy(handle)
    return [x.detach().cpu() for x in (out, q.grad, k.grad, v.grad)], path


def _csr(mat, bs):
    full = np.repeat(np.repeat(mat != 0, bs, 0), bs, 1)
    sm = full.sum(1).astype(np.int32)
    return sm, np.concatenate([[0], np.cumsum(sm)]).astype(np.int32), np.nonzero(full)[1].astype(np.int32)


# a wavefront to a strip and four; past one wavefront's registers at d = 64 (20 tiles); the two sweeps (34)
@pytest.mark.parametrize("d", [32, 64])
@pytest.mark.parametrize("L,route", [(96, "module"), (640, "module"), (640, "strided"), (640, "abi"), (1088, "module")])
@pytest.mark.parametrize("which", ["q", "k", "v", "do"])
def test_infinities_nan_and_the_largest_floats(which, L, route, d):
    """Against the element kernels, whose sums are fp32 throughout, on the same pattern and operands.  (The two sweeps start a
    logit's chain from the row's maximum: 2^120 less itself is rounding noise of 2^97 there.)"""
    mat = workloads.band_random_block_mask(L // 32, 1, extra_frac=1.0, seed=L + d)
    for value in LIMITS[: 3 if which in ("q", "k") and L > 1024 else 5]:
        t = _special(which, value, 2, L, d)
        got, path = _run_sparse(t, mat, 32, False, route)
        want, path_e = _run_sparse(t, mat, 32, True, route)
        assert (path, path_e) == (1, 2)
        _compare(got, want, which, value, L + d)


@pytest.mark.parametrize("which", ["q", "k", "v", "do"])
def test_infinities_in_the_tiles_of_element_patterns(which):
    """Against the element kernels; an absent entry of a tile counts there with probability 0, which times an infinity is NaN,
    so only what no infinity is multiplied with compares: the output for q and k, the largest floats for V and dO."""
    L, d = 1056, 32
    i, g = np.arange(L), np.random.default_rng(1)
    mat = ((g.random((L, L)) < 35 / L) | (abs(i[:, None] - i[None, :]) <= 24)).astype(np.float32)
    for value in LIMITS[:3] if which in ("q", "k") else LIMITS[3:]:
        t = _special(which, value, 2, L, d)
        got, path = _run_sparse(t, mat, 1, False, "module")
        want, path_e = _run_sparse(t, mat, 1, True, "module")
        assert (path, path_e) == (3, 2)
        _compare(got, want, which, value, L + d, outputs=1 if which in ("q", "k") else 4)


# register-resident with four wavefronts and with eight, two sweeps; feature-major operands
@pytest.mark.parametrize("d,L,views", [(32, 96, True), (32, 1024, False), (32, 1088, True), (32, 2080, True), (32, 2080, False),
                                       (64, 96, True), (64, 1088, True)])
@pytest.mark.parametrize("which", ["q", "k", "v", "do"])
def test_dense_phase_infinities_nan_and_the_largest_floats(which, L, d, views):
    """Against the same steps as torch runs them in fp32.  (Two sweeps and logits of 2^120: see above.)"""
    for value in LIMITS[: 3 if which in ("q", "k") and L > 2048 else 5]:
        t = _special(which, value, 1, L, d)
        cpp = spion_amd.Attention._cuda_compile_module()
        mod = spion_amd.CUDAAttention(dict(head_dim=d, num_head=1, max_seq_len=L, batch_size=1), cpp, cpp.init(d, L, 1))
        mod.reads_views = views
        q, k, v = (t[n].cuda().requires_grad_() for n in "qkv")
        out, _ = mod(q, k, v, torch.ones(1, L, device="cuda"))
        out.backward(t["do"].cuda())
        cpp.destroy(mod.attn_handle)
        Q, K, V, dO = (t[n].cuda()[0, 0] for n in ("q", "k", "v", "do"))
        s = (Q * (d ** -0.5 * LOG2E)) @ K.t()
        e = torch.exp2(s - torch.fmax(s, torch.tensor(-10.0 * LOG2E, device="cuda")).amax(-1, keepdim=True))
        P = e / e.sum(-1, keepdim=True)
        O = P @ V
        ds = (dO @ V.t() - (dO * O).sum(-1, keepdim=True)) * P
        want = [O, ds @ K * d ** -0.5, ds.t() @ Q * d ** -0.5, P.t() @ dO]
        _compare([x.detach()[0, 0].cpu() for x in (out, q.grad, k.grad, v.grad)], [x.cpu() for x in want], which, value, L + d)


@pytest.mark.parametrize("d", [32, 64])
@pytest.mark.parametrize("power", [-100, -112, -117])
def test_gradients_near_the_smallest_floats(d, power):
    """An incoming gradient of 2^-112 or 2^-117: the third part of its elements is subnormal or lost, up to 2^-16 of an element.
    The gradients keep the accuracy that they have at any other scale (2-norms; at most L roundings of 2^-24 that add up
    like a random walk, with a margin of two)."""
    L, bs = 256, 32
    mat = workloads.band_random_block_mask(L // bs, 1, extra_frac=0.5, seed=d)
    t = _special("do", 0.0, 2, L, d)
    t["do"] = t["do"] * 2.0 ** power
    got, _ = _run_sparse(t, mat, bs, False, "module")
    pat = torch.from_numpy(mat).double().repeat_interleave(bs, 0).repeat_interleave(bs, 1)
    ref = [t[n].double().requires_grad_() for n in "qkv"]
    osa.dense_masked_attention(*ref, pat)[0].backward(t["do"].double())
    for name, x, y in zip(NAMES[1:], got[1:], ref):
        err = float((x.double() - y.grad).norm() / y.grad.norm())
        assert err < 2 * L ** 0.5 * EPS, (name, err)


def improbable(H, L, d, seed):
    """Normal operands [1, H, L, d] in which one key, L/2 + 1, has a logit of -80 in every row (a probability of about 2^-122),
    and the gradients of one query, L/2 - 5, are 2^-118 of the others'."""
    g = torch.Generator().manual_seed(seed)
    t = dict(zip(("q", "k", "v", "do"), (torch.randn(1, H, L, d, generator=g) for _ in range(4))))
    t["q"][..., 0] = 4.0
    t["k"][..., 0] = 0.0
    t["k"][:, :, L // 2 + 1] = 0.0
    t["k"][:, :, L // 2 + 1, 0] = -80.0 * d ** 0.5 / 4.0
    t["do"][:, :, L // 2 - 5] *= 2.0 ** -118
    return t


def compare_by_element(t, p, out, grads, d):
    """Gradients [H, L, d] against float64 steps from the probabilities [H, L, L] and the output the kernels left, each element
    within the roundings of its own terms: `n + 8` of the magnitudes of a sum of n, as in `_bounds`, two for the product
    with a probability, and 2^-149 a term where a product is subnormal."""
    L = p.shape[-1]
    rnd, tr = lambda n: (n + 8) * EPS, lambda x: x.transpose(-1, -2)
    q, k, v, do = (t[n][0].double() for n in ("q", "k", "v", "do"))
    p, out = p.double().cpu(), out.double().cpu()
    assert 2.0 ** -126 < float(p[..., L // 2 + 1].max()) < 2.0 ** -120
    mag = do.abs() @ tr(v).abs() + (do * out).abs().sum(-1, keepdim=True)
    ds = p * (do @ tr(v) - (do * out).sum(-1, keepdim=True))
    eds = (rnd(d) + 2 * EPS) * p * mag + 2.0 ** -149
    want = [ds @ k * d ** -0.5, tr(ds) @ q * d ** -0.5, tr(p) @ do]
    bound = [d ** -0.5 * (eds @ k.abs() + rnd(L) * ds.abs() @ k.abs()), d ** -0.5 * (tr(eds) @ q.abs() + rnd(L) * tr(ds).abs() @ q.abs()),
             rnd(L) * tr(p) @ do.abs()]
    for name, x, y, e in zip(NAMES[1:], grads, want, bound):
        worst = float(((x.double().cpu() - y).abs() / (e + L * 2.0 ** -149)).max())
        assert worst <= 1.0, f"{name}: {worst} of the bound"


# a wavefront to a strip and four
@pytest.mark.parametrize("d", [32, 64])
@pytest.mark.parametrize("L,route", [(96, "module"), (640, "module"), (640, "strided"), (640, "abi")])
def test_a_small_row_among_ordinary_ones(L, route, d):
    H, bs = 2, 32
    t = improbable(H, L, d, L + d)
    mat = np.ones((L // bs, L // bs), dtype=np.float32)
    if route == "abi":
        abi = SparseABI(d, L, H, bs, with_mask=True)
        abi.set_pattern(*_csr(mat, bs))
        q, k, v, do = (t[n][0].cuda() for n in ("q", "k", "v", "do"))
        out, p = abi.forward(q, k, v, torch.zeros(H, L, device="cuda"))
        grads, path = abi.backward(q, k, v, p, do), abi.last_path()
        abi.close()
    else:
        cpp = spion_amd.Attention._blockcuda_compile_module()
        handle = cpp.init(d, L, H, bs)
        mod = spion_amd.CUDABlockAttention(dict(head_dim=d, num_head=H, max_seq_len=L, batch_size=1, block_size=bs), cpp, handle)
        place = lambda x: x.cuda().transpose(1, 2).contiguous().transpose(1, 2) if route == "strided" else x.cuda()
        leaves = [place(t[n]).requires_grad_() for n in "qkv"]
        out, p = mod(*leaves, torch.ones(1, L, device="cuda"), torch.from_numpy(mat).cuda())
        out.backward(t["do"].cuda())
        grads, path = [x.grad[0] for x in leaves], _lib.core().spion_last_path(handle)
        out, p = out.detach()[0], p.detach()
        cpp.destroy(handle)
    assert path == 1
    compare_by_element(t, p.reshape(H, L, L), out, grads, d)
