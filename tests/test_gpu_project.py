"""Projection kernels (spion_project_*) and the layer that runs on them, against float64 (on a GPU only)."""
import ctypes

import pytest
import torch

import spion_amd
from spion_amd import _lib, workloads

pytestmark = pytest.mark.gpu


def _ptrs(ts):
    return (ctypes.c_void_p * len(ts))(*[t.data_ptr() for t in ts])


def _check(got, a, b, extra=None, pieces=1):
    """got = a @ b (+ extra): every fp32 accumulation step rounds by at most 2^-24 of the running sum of magnitudes; a
    reduction index takes 12/32 matrix instructions, each of which adds once to the accumulator, the six dropped or
    rounded partial products of an element pair stay below 2^-24 of it, and pieces are added once more each."""
    a, b = a.double(), b.double()
    ref, mag = a @ b, a.abs() @ b.abs()
    if extra is not None:
        ref, mag = ref + extra.double(), mag + extra.double().abs()
    steps = 12 * a.shape[-1] / 32 + pieces + 2
    assert bool(((got.double() - ref).abs() <= steps * 2.0 ** -24 * mag).all()), float(((got.double() - ref).abs() / mag).max())


# tile edges (64 and 128), odd numbers of 32-blocks, one segment and three, many pieces, the 128 x 128 tiles
@pytest.mark.parametrize("rows,dim,n,segs", [(32, 32, 32, 1), (64, 32, 32, 3), (96, 64, 32, 2), (1056, 96, 96, 3), (4000, 64, 64, 3),
                                             (65536, 64, 64, 1), (160, 160, 352, 1), (8192, 512, 512, 3), (65536, 256, 128, 3)])
def test_projection_kernels_match_float64(rows, dim, n, segs):
    g = torch.Generator().manual_seed(rows + dim)
    x = torch.randn(rows, dim, generator=g).cuda()
    w = [torch.randn(n, dim, generator=g).cuda() for _ in range(segs)]
    b = [torch.randn(n, generator=g).cuda() for _ in range(segs)]
    dy = (torch.randn(rows, segs * n, generator=g) + 0.5).cuda()  # a mean: the column sums grow
    core, stream = _lib.core(), torch.cuda.current_stream().cuda_stream
    y = torch.full((rows + 1, segs * n), 7.0, device="cuda")
    assert core.spion_project_forward(x.data_ptr(), _ptrs(w), _ptrs(b), y.data_ptr(), rows, n, segs, dim, stream) == 0
    assert bool((y[rows] == 7.0).all())  # nothing past the end
    W, bias = torch.cat(w), torch.cat(b)
    _check(y[:rows], x, W.t(), bias)
    dx = torch.full((rows + 1, dim), 7.0, device="cuda")
    assert core.spion_project_backward_input(dy.data_ptr(), _ptrs(w), dx.data_ptr(), rows, n, segs, dim, stream) == 0
    assert bool((dx[rows] == 7.0).all())
    _check(dx[:rows], dy, W)
    N = segs * n
    got = []
    for _ in range(2):
        dw = torch.full((N * dim + 4,), 7.0, device="cuda")
        db = torch.full((N + 4,), 7.0, device="cuda")
        ws = torch.empty(core.spion_project_workspace(rows, N, dim), device="cuda")
        assert core.spion_project_backward_weight(dy.data_ptr(), x.data_ptr(), dw.data_ptr(), db.data_ptr(), ws.data_ptr(), rows,
                                                  N, dim, stream) == 0
        assert bool((dw[N * dim:] == 7.0).all()) and bool((db[N:] == 7.0).all())
        got.append((dw[: N * dim].view(N, dim), db[:N]))
    _check(got[0][0], dy.t(), x, pieces=256)
    _check(got[0][1][:, None], dy.t(), torch.ones(rows, 1, device="cuda"), pieces=256 + rows)
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


# one launch for dX, dW and db (and its limits: one piece, ragged pieces, tiles past the outputs), 128 x 128 tiles of dX (two calls)
@pytest.mark.parametrize("rows,dim,n,segs", [(32, 32, 32, 1), (96, 64, 32, 2), (1056, 96, 96, 3), (2080, 64, 64, 3), (65536, 64, 64, 1),
                                             (160, 160, 352, 1), (65536, 256, 128, 3)])
def test_joint_backward_has_the_bits_of_the_two_calls(rows, dim, n, segs):
    g = torch.Generator().manual_seed(rows + dim)
    x = torch.randn(rows, dim, generator=g).cuda()
    w = [torch.randn(n, dim, generator=g).cuda() for _ in range(segs)]
    N = segs * n
    dy = (torch.randn(rows, N, generator=g) + 0.5).cuda()
    core, stream = _lib.core(), torch.cuda.current_stream().cuda_stream
    ws = torch.empty(core.spion_project_workspace(rows, N, dim), device="cuda")
    outs = [[torch.full((size + 4,), 7.0, device="cuda") for size in (rows * dim, N * dim, N)] for _ in range(2)]
    dx, dw, db = (t.data_ptr() for t in outs[0])
    assert core.spion_project_backward(dy.data_ptr(), _ptrs(w), x.data_ptr(), dx, dw, db, ws.data_ptr(), rows, n, segs, dim, stream) == 0
    dx, dw, db = (t.data_ptr() for t in outs[1])
    assert core.spion_project_backward_input(dy.data_ptr(), _ptrs(w), dx, rows, n, segs, dim, stream) == 0
    assert core.spion_project_backward_weight(dy.data_ptr(), x.data_ptr(), dw, db, ws.data_ptr(), rows, N, dim, stream) == 0
    for a, b in zip(*outs):
        assert torch.equal(a, b) and bool((a[-4:] == 7.0).all())
    for args in ((None, x.data_ptr(), dx), (_ptrs(w), None, dx), (_ptrs(w), x.data_ptr(), None)):
        assert core.spion_project_backward(dy.data_ptr(), *args, dw, db, ws.data_ptr(), rows, n, segs, dim, stream) != 0
        _lib.core().spion_clear_error()


def _kinds(x):
    return torch.isposinf(x) + 2 * torch.isneginf(x) + 3 * torch.isnan(x)


# narrow and wide tiles; many pieces of the weight gradient's sum
@pytest.mark.parametrize("rows,dim,n", [(96, 64, 32), (16384, 64, 64), (8192, 512, 512)])
@pytest.mark.parametrize("which", ["x", "w", "dy"])
def test_infinities_nan_and_the_largest_floats(rows, dim, n, which):
    """One special element: the same results infinite and NaN as torch's fp32 products give, finite ones to the accuracy that
    they have without it.  Beside a finite one everything is a sixteenth, so that no product with it overflows."""
    g = torch.Generator().manual_seed(rows)
    core, stream = _lib.core(), torch.cuda.current_stream().cuda_stream
    for value in (float("inf"), -float("inf"), float("nan"), 2.0 ** 128 - 2.0 ** 104, -(2.0 ** 128 - 2.0 ** 119)):
        t = {k: torch.randn(*s, generator=g).cuda() for k, s in dict(x=(rows, dim), w=(n, dim), dy=(rows, n)).items()}
        if 1.0 < abs(value) < float("inf"):
            t = {k: v / 16 for k, v in t.items()}
        t[which][5, 7] = value
        x, w, dy, b = t["x"], t["w"], t["dy"], torch.randn(n, device="cuda")
        y, dx, dw, db = (torch.empty_like(v) for v in (dy, x, w, b))
        ws = torch.empty(core.spion_project_workspace(rows, n, dim), device="cuda")
        assert core.spion_project_forward(x.data_ptr(), _ptrs([w]), _ptrs([b]), y.data_ptr(), rows, n, 1, dim, stream) == 0
        assert core.spion_project_backward_input(dy.data_ptr(), _ptrs([w]), dx.data_ptr(), rows, n, 1, dim, stream) == 0
        assert core.spion_project_backward_weight(dy.data_ptr(), x.data_ptr(), dw.data_ptr(), db.data_ptr(), ws.data_ptr(), rows,
                                                  n, dim, stream) == 0
        for name, got, a, c, extra in (("y", y, x, w.t(), b), ("dx", dx, dy, w, None), ("dw", dw, dy.t(), x, None)):
            ref = a @ c if extra is None else a @ c + extra
            assert torch.equal(_kinds(got), _kinds(ref)), (name, value)
            ok = torch.isfinite(ref)
            mag = a.abs().double() @ c.abs().double()
            err = (got.double() - ref.double()).abs()
            terms = min(a.shape[1], 1024) + 256  # a piece's terms one by one on both sides, and the pieces
            assert bool((err[ok] <= 2 * terms * 2.0 ** -24 * mag[ok] + 2.0 ** -20).all()), (name, value)


def test_products_near_the_smallest_floats():
    """Operands of 2^-117: their third parts are subnormal or lost, up to 2^-16 of an element."""
    rows, dim, n = 2048, 64, 64
    g = torch.Generator().manual_seed(1)
    core, stream = _lib.core(), torch.cuda.current_stream().cuda_stream
    x, w = torch.randn(rows, dim, generator=g).cuda(), torch.randn(n, dim, generator=g).cuda()
    dy = (torch.randn(rows, n, generator=g) * 2.0 ** -117).cuda()
    dx, dw, db = torch.empty_like(x), torch.empty_like(w), torch.empty(n, device="cuda")
    ws = torch.empty(core.spion_project_workspace(rows, n, dim), device="cuda")
    assert core.spion_project_backward_input(dy.data_ptr(), _ptrs([w]), dx.data_ptr(), rows, n, 1, dim, stream) == 0
    assert core.spion_project_backward_weight(dy.data_ptr(), x.data_ptr(), dw.data_ptr(), db.data_ptr(), ws.data_ptr(), rows, n,
                                              dim, stream) == 0
    for got, ref in ((dx, dy.double() @ w.double()), (dw, dy.double().t() @ x.double())):
        assert float((got.double() - ref).norm() / ref.norm()) < 1e-6  # some tens of roundings of 2^-24


def test_rows_past_a_quarter_of_the_int_range():
    """Row indices from 2^29 on are rows of the matrix like any other: the last 64 of 2^29 + 32 rows."""
    rows = 2 ** 29 + 32
    if torch.cuda.mem_get_info()[0] < 160 * 2 ** 30:
        pytest.skip("needs 140 GB of device memory")
    x = torch.zeros(rows, 32, device="cuda")
    tail = torch.randn(64, 32, generator=torch.Generator().manual_seed(1)).cuda()
    x[-64:] = tail
    w, b = torch.randn(32, 32, device="cuda"), torch.randn(32, device="cuda")
    y = torch.empty(rows, 32, device="cuda")
    core, stream = _lib.core(), torch.cuda.current_stream().cuda_stream
    assert core.spion_project_forward(x.data_ptr(), _ptrs([w]), _ptrs([b]), y.data_ptr(), rows, 32, 1, 32, stream) == 0
    _check(y[-64:], tail, w.t(), b)
    assert core.spion_project_backward_input(x.data_ptr(), _ptrs([w]), y.data_ptr(), rows, 32, 1, 32, stream) == 0
    _check(y[-64:], tail, w)
    del x, y
    torch.cuda.empty_cache()


def test_weight_gradient_of_one_signed_data_keeps_fp32_accuracy():
    """All operands just above a bf16 number, summed over many rows: the small partial products then share a sign and must
    not be lost against the large sum."""
    rows = 131072
    dy = torch.full((rows, 32), 1.0 + 3 * 2.0 ** -16, device="cuda")
    x = torch.full((rows, 32), 1.0 + 3 * 2.0 ** -16, device="cuda")
    core, stream = _lib.core(), torch.cuda.current_stream().cuda_stream
    dw, db = torch.empty(32, 32, device="cuda"), torch.empty(32, device="cuda")
    ws = torch.empty(core.spion_project_workspace(rows, 32, 32), device="cuda")
    assert core.spion_project_backward_weight(dy.data_ptr(), x.data_ptr(), dw.data_ptr(), db.data_ptr(), ws.data_ptr(), rows, 32, 32,
                                              stream) == 0
    ref = rows * (1.0 + 3 * 2.0 ** -16) ** 2
    assert float((dw.double() - ref).abs().max()) / ref < 2e-6  # 512 rows a piece and 256 pieces: about 30 roundings of 2^-24


@pytest.mark.parametrize("heads", [1, 2, 5])
def test_key_penalty_is_the_modules_expression(heads):
    mask = workloads.valid_length_mask(3, 96, 10, 96, seed=1).cuda()
    mask[0, 0] = 0.25
    pen = torch.empty(3, heads * 96, device="cuda")
    assert _lib.core().spion_key_penalty(mask.data_ptr(), pen.data_ptr(), 3, heads, 96, torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(pen, 1e6 * (1.0 - mask.repeat(1, heads)))


@pytest.mark.parametrize("heads,d,L,masked", [(2, 32, 256, False), (1, 32, 288, True), (4, 64, 128, True), (3, 32, 160, False)])
def test_layer_in_one_call_matches_its_steps(heads, d, L, masked):
    """The compiled whole-layer path against the same layer run step by step (torch projections), with and without
    gradients; a frozen weight gets none; a hook on a submodule switches to the steps."""
    if _lib.autograd_node() is None:
        pytest.skip("SPION_PY_NODE=1")
    B, bs = 3, 32
    cfg = dict(head_dim=d, num_head=heads, max_seq_len=L, batch_size=B, block_size=bs, transformer_dim=96, attention_dropout=0.0,
               task="lra-text" if masked else "lra-image")
    torch.manual_seed(heads)
    layer = spion_amd.Attention(cfg, inference=True).cuda()
    layer.reconstruct_for_blocksparse(cfg)
    mat = torch.from_numpy(workloads.band_random_block_mask(L // bs, 1, extra_frac=0.2, seed=3)).cuda()
    mask = workloads.valid_length_mask(B, L, L // 2, L, seed=5).cuda()
    x, dy = torch.randn(B, L, 96, device="cuda", requires_grad=True), torch.randn(B, L, 96, device="cuda")

    def run():
        x.grad = None
        layer.zero_grad(set_to_none=True)
        y, p = layer(x, mask, mat)
        y.backward(dy)
        return [y.detach(), p] + [x.grad] + [t.grad for t in layer.parameters()]

    fused = [t.detach() if isinstance(t, torch.Tensor) else t for t in run()]
    with torch.no_grad():
        y0, p0 = layer(x, mask, mat)
    assert torch.equal(y0, fused[0]) and (masked or torch.equal(p0, fused[1]))
    calls = []
    hook = layer.ff.register_forward_hook(lambda *a: calls.append(1))
    steps = [t.detach() if isinstance(t, torch.Tensor) else t for t in run()]
    assert calls
    hook.remove()
    for a, b in zip(fused, steps):
        if isinstance(a, int):
            assert a == b == 0
            continue
        assert a.shape == b.shape
        assert float((a - b).norm() / b.norm()) < 2e-6  # both fp32 throughout
    layer.W_k.weight.requires_grad_(False)
    again = run()
    assert layer.W_k.weight.grad is None
    assert torch.equal(again[2], fused[2])


@pytest.mark.parametrize("how", ["global hook", "global pre-hook", "own forward"])
def test_layer_runs_its_modules_when_they_are_watched(how):
    """Hooks on all modules see the core and the output projection, and a forward set on an instance runs."""
    B, L = 2, 64
    cfg = dict(head_dim=32, num_head=2, max_seq_len=L, batch_size=B, block_size=32, transformer_dim=96, attention_dropout=0.0,
               task="lra-image")
    layer = spion_amd.Attention(cfg, inference=True).cuda()
    layer.reconstruct_for_blocksparse(cfg)
    args = (torch.randn(B, L, 96, device="cuda"), torch.ones(B, L, device="cuda"), torch.eye(2, device="cuda"))
    plain = layer(*args)[0]
    seen, handle = [], None
    if how == "own forward":
        for m in (layer.ff, layer.block_attn):
            m.forward = lambda *a, m=m: (seen.append(m), type(m).forward(m, *a))[1]
    elif how == "global hook":
        handle = torch.nn.modules.module.register_module_forward_hook(lambda m, i, o: seen.append(m) and None)
    else:
        handle = torch.nn.modules.module.register_module_forward_pre_hook(lambda m, i: seen.append(m) and None)
    try:
        watched = layer(*args)[0]
    finally:
        if handle:
            handle.remove()
    assert layer.ff in seen and layer.block_attn in seen
    assert float((watched - plain).detach().norm() / plain.detach().norm()) < 2e-6
    if handle:
        seen.clear()
        assert torch.equal(layer(*args)[0], plain) and not seen


@pytest.mark.parametrize("outputs", [48, 64, 160])
def test_layer_with_a_replaced_output_projection(outputs):
    """Another width of the output projection: on the kernels where it is a multiple of 32, torch's steps where not."""
    B, L = 2, 64
    cfg = dict(head_dim=32, num_head=2, max_seq_len=L, batch_size=B, block_size=32, transformer_dim=96, attention_dropout=0.0,
               task="lra-image")
    layer = spion_amd.Attention(cfg, inference=True)
    layer.ff = torch.nn.Linear(64, outputs)
    layer = layer.cuda()
    layer.reconstruct_for_blocksparse(cfg)
    x, mat = torch.randn(B, L, 96, device="cuda", requires_grad=True), torch.eye(2, device="cuda")
    seen = []
    ones = torch.ones(B, L, device="cuda")
    y, _ = layer(x, ones, mat)
    layer.block_attn.register_forward_hook(lambda m, i, o: seen.append(o[0].detach()))
    y2, _ = layer(x, ones, mat)
    ref = torch.nn.functional.linear(layer.combine_heads(seen[0]).double(), layer.ff.weight.double(), layer.ff.bias.double())
    assert y.shape == (B, L, outputs)
    for t in (y, y2):
        assert float((t.detach().double() - ref.detach()).norm() / ref.detach().norm()) < 2e-6
    y.sum().backward()
    assert layer.ff.weight.grad.shape == (outputs, 64)


@pytest.mark.parametrize("which", ["W_q", "W_v", "ff"])
def test_layer_with_a_replaced_projection_that_does_not_fit_raises(which):
    B, L = 2, 64
    cfg = dict(head_dim=32, num_head=2, max_seq_len=L, batch_size=B, block_size=32, transformer_dim=96, attention_dropout=0.0,
               task="lra-image")
    layer = spion_amd.Attention(cfg, inference=True)
    setattr(layer, which, torch.nn.Linear(32, 96) if which == "ff" else torch.nn.Linear(96, 32))
    layer = layer.cuda()
    layer.reconstruct_for_blocksparse(cfg)
    with pytest.raises(RuntimeError):
        layer(torch.randn(B, L, 96, device="cuda"), torch.ones(B, L, device="cuda"), torch.eye(2, device="cuda"))


def test_layer_with_a_core_of_other_heads_raises():
    B, L = 2, 64
    cfg = dict(head_dim=32, num_head=2, max_seq_len=L, batch_size=B, block_size=32, transformer_dim=96, attention_dropout=0.0,
               task="lra-image")
    layer = spion_amd.Attention(cfg, inference=True).cuda()
    layer.reconstruct_for_blocksparse(dict(cfg, num_head=4))
    with pytest.raises(ValueError, match="does not match the handle"):
        layer(torch.randn(B, L, 96, device="cuda"), torch.ones(B, L, device="cuda"), torch.eye(2, device="cuda"))


@pytest.mark.skipif(torch.cuda.device_count() < 2, reason="needs two GPUs")
def test_layer_runs_on_its_inputs_device():
    """A layer on another GPU than the current one, as torch's linear layers allow."""
    B, L = 2, 64
    cfg = dict(head_dim=32, num_head=2, max_seq_len=L, batch_size=B, block_size=32, transformer_dim=96, attention_dropout=0.0,
               task="lra-text")
    args = (torch.randn(B, L, 96, device="cuda:1"), torch.ones(B, L, device="cuda:1"), torch.eye(2, device="cuda:1"))
    with torch.cuda.device(1):
        layer = spion_amd.Attention(cfg, inference=True).cuda()
        layer.reconstruct_for_blocksparse(cfg)
        there = layer(*args)[0]
    with torch.cuda.device(0):
        here = layer(*args)[0]
        here.sum().backward()
    assert here.device == there.device and torch.equal(here, there)


# narrow and wide tiles; fewer and more penalties than a work-group's 256 threads, several rounds of the most work-groups
@pytest.mark.parametrize("rows,dim,B,H,L", [(32, 32, 1, 1, 32), (96, 64, 3, 2, 32), (4096, 64, 2, 8, 2048), (32768, 256, 16, 4, 2048),
                                            (65536, 32, 64, 16, 1024)])
def test_penalties_made_beside_the_projections(rows, dim, B, H, L):
    """Both outputs bit for bit as from launches of their own."""
    g = torch.Generator(device="cuda").manual_seed(rows)
    x = torch.randn(rows, dim, generator=g, device="cuda")
    w = [torch.randn(64, dim, generator=g, device="cuda") for _ in range(3)]
    b = [torch.randn(64, generator=g, device="cuda") for _ in range(3)]
    mask = torch.rand(B, L, generator=g, device="cuda").round()
    mask[0, 0] = 0.25
    core, stream = _lib.core(), torch.cuda.current_stream().cuda_stream
    y, y2 = (torch.full((rows, 192), float("nan"), device="cuda") for _ in range(2))
    pen, pen2 = (torch.full((B * H, L), float("nan"), device="cuda") for _ in range(2))
    assert core.spion_project_forward(x.data_ptr(), _ptrs(w), _ptrs(b), y.data_ptr(), rows, 64, 3, dim, stream) == 0
    assert core.spion_key_penalty(mask.data_ptr(), pen.data_ptr(), B, H, L, stream) == 0
    assert core.spion_project_forward_keys(x.data_ptr(), _ptrs(w), _ptrs(b), y2.data_ptr(), rows, 64, 3, dim, mask.data_ptr(),
                                           pen2.data_ptr(), B, H, L, stream) == 0
    assert torch.equal(y, y2) and torch.equal(pen, pen2)
    assert core.spion_project_forward_keys(x.data_ptr(), _ptrs(w), _ptrs(b), y2.data_ptr(), rows, 64, 3, dim, None, None, B, H, L,
                                           stream) != 0
    with pytest.raises(_lib.SpionLibraryError, match="null mask"):
        _lib.check_error("projection")
