"""The remainder kernels by ranges (remainder_kernels.h) at the edges of their ranges, batches and work-groups, against float64
on some of the heads (on a GPU only)."""
import pytest
import torch

import spion_amd
from spion_amd import _lib

pytestmark = pytest.mark.gpu


def _pattern(L, gen):
    """A window and a few random columns; row 7 and row L - 3 with many entries in one range (more than a batch), a column that
    every third row has, an empty row, a column of the last range that no row has."""
    i = torch.arange(L, device="cuda")
    m = (torch.rand(L, L, generator=gen, device="cuda") < 14 / L).float()
    m[(i[:, None] - i[None, :]).abs() <= 40] = 1.0
    m[7, 1:500:3] = 1.0
    m[L - 3, 100:500:7] = 1.0
    m[::3, 450] = 1.0
    m[5] = 0.0
    m[:, L - 2] = 0.0
    return m


def _reference(q, k, v, do, pattern, valid):
    q, k, v = (t.double().requires_grad_() for t in (q, k, v))
    s = q @ k.transpose(-1, -2).contiguous() / q.shape[-1] ** 0.5
    if valid is not None:
        s = s - 1e6 * (1.0 - valid.double())[:, None, :]
    p = torch.softmax(s * pattern, -1) * pattern
    o = p @ v
    o.backward(do.double())
    return p.detach(), o.detach(), q.grad, k.grad, v.grad


def _module(B, H, L, masked):
    cfg = dict(head_dim=32, num_head=H, max_seq_len=L, batch_size=B, block_size=1)
    load, cls = (("_blockcuda_mask_compile_module", spion_amd.CUDABlockMaskAttention) if masked else
                 ("_blockcuda_compile_module", spion_amd.CUDABlockAttention))
    cpp = getattr(spion_amd.Attention, load)()
    handle = cpp.init(32, L, B * H, 1)
    return cpp, handle, cls(cfg, cpp, handle)


# one range; a second one of 32 rows; work-groups of 256 rows whose last is partial; work-groups of 512, the last partial; nine ranges
@pytest.mark.parametrize("B,H,L,masked", [(32, 2, 512, False), (24, 2, 544, True), (14, 2, 1056, False), (35, 2, 1056, True),
                                          (35, 2, 1056, False), (32, 2, 2048, False), (24, 2, 4128, True)])
@pytest.mark.parametrize("views", [False, True])
def test_ranges_and_batches(B, H, L, masked, views):
    gen = torch.Generator(device="cuda").manual_seed(L + B)
    pattern = _pattern(L, gen)
    shape = (B, L, H, 32) if views else (B, H, L, 32)
    make = lambda: torch.randn(*shape, generator=gen, device="cuda")
    q, k, v, do = (make().transpose(1, 2) if views else make() for _ in range(4))
    leaves = [t.requires_grad_() for t in (q, k, v)]
    i = torch.arange(L, device="cuda")
    valid = (i[None, :] < torch.randint(L // 2, L + 1, (B, 1), generator=gen, device="cuda")).float() if masked else \
        torch.ones(B, L, device="cuda")
    cpp, handle, module = _module(B, H, L, masked)
    out, p = module(*leaves, valid, pattern)
    out.backward(do)
    torch.cuda.synchronize()
    assert _lib.core().spion_last_path(handle) == 3
    assert _lib.core().spion_debug_counter(handle, 3) == 1
    where = pattern.bool()
    p = None if masked else p.detach().reshape(B, H, -1)  # the masked module does not return it
    for b, h in ((0, 0), (B // 2, H - 1), (B - 1, H - 1)):
        at = lambda t: t.detach()[b, h][None]
        ref = _reference(at(q), at(k), at(v), at(do), pattern.double()[None], valid[b][None] if masked else None)
        got = (None if masked else p[b, h],) + tuple(at(t) for t in (out, q.grad, k.grad, v.grad))
        for name, x, y in zip(("P", "out", "dQ", "dK", "dV"), got, (ref[0][0][where],) + ref[1:]):
            if x is None:
                continue
            # A hundred to some thousand terms each, of unlike signs: their roundings, 2^-24 each, add up as the terms do, to a few
            # 2^-24 of a typical element (2.3e-7 seen), ten times that for the furthest of 30,000 to 400,000 (2.6e-6 seen).
            diff, typical = x.double() - y, y.pow(2).mean().sqrt()
            assert float(diff.pow(2).mean().sqrt() / typical) <= 1e-6, f"{name}, head {(b, h)}"
            worst = float((diff.abs() / (y.abs() + typical)).max())
            assert worst <= 1e-5, f"{name}, head {(b, h)}: {worst}"
    cpp.destroy(handle)


def test_infinities_stay_in_their_rows():
    """The slots of a batch that hold no entry read a row of zeros, and tiles are taken by their entries: an infinity reaches the
    rows that have its column and no other."""
    B, H, L, far = 16, 2, 1024, 900
    gen = torch.Generator(device="cuda").manual_seed(1)
    pattern = _pattern(L, gen)
    q, k, v, do = (torch.randn(B, H, L, 32, generator=gen, device="cuda") for _ in range(4))
    q[..., far, 3] = v[..., far, 3] = do[..., far, 5] = float("inf")
    q, k, v = (t.requires_grad_() for t in (q, k, v))
    cpp, handle, module = _module(B, H, L, False)
    out, p = module(q, k, v, torch.ones(B, L, device="cuda"), pattern)
    out.backward(do)
    assert _lib.core().spion_last_path(handle) == 3
    assert _lib.core().spion_debug_counter(handle, 3) == 1
    # Q of row far: that row; V: the rows that have the column; dO of row far: as Q.  dK takes {dS, P} of all of them, dV those of row far
    bad_rows = pattern[:, far] > 0
    bad_rows[far] = True
    exactly = lambda t, reached: torch.equal(torch.isfinite(t).all(-1), (~reached).expand(B, H, L))
    assert exactly(out, bad_rows) and exactly(q.grad, bad_rows)
    assert exactly(k.grad, (pattern[bad_rows] > 0).any(0)) and exactly(v.grad, pattern[far] > 0)
    cpp.destroy(handle)


@pytest.mark.parametrize("kind", ["window", "scattered"])
def test_rows_without_entries_take_nothing_from_infinities(kind):
    """A row of the pattern without entries: its gradient of Q stays zero whatever its dO (and dO . O) is."""
    B, H, L = 16, 2, 1024
    gen = torch.Generator(device="cuda").manual_seed(8)
    pattern = _pattern(L, gen) if kind == "window" else _scattered(L, gen)
    empty = (pattern.sum(1) == 0).nonzero()[:, 0].tolist()
    assert empty
    if kind == "window":  # neither do the block row's dense tiles hold the row
        for i in empty:
            pattern[i // 32 * 32: i // 32 * 32 + 32] *= (torch.rand(32, L, generator=gen, device="cuda") < 0.1).float()
    q, k, v, do = (torch.randn(B, H, L, 32, generator=gen, device="cuda") for _ in range(4))
    do[..., empty, 5] = float("inf")
    q, k, v = (t.requires_grad_() for t in (q, k, v))
    cpp, handle, module = _module(B, H, L, False)
    out, p = module(q, k, v, torch.ones(B, L, device="cuda"), pattern)
    out.backward(do)
    assert _lib.core().spion_debug_counter(handle, 3) == 1
    assert (out[..., empty, :] == 0).all() and (q.grad[..., empty, :] == 0).all()
    for t in (out, q.grad, k.grad, v.grad):
        assert torch.isfinite(t).all()
    cpp.destroy(handle)


def _holed(L, half, gen):
    """A window of the given half width that lacks a fifth of its entries, and random columns; half 0: whole and holed tiles that
    hold less than half of the entries."""
    i = torch.arange(L, device="cuda")
    pattern = (torch.rand(L, L, generator=gen, device="cuda") < (0.02 if half else 0.06)).float()
    holes = (torch.rand(L, L, generator=gen, device="cuda") < 0.8).float()
    if half:
        near = (i[:, None] - i[None, :]).abs() <= half
        return torch.where(near, holes, pattern)
    for n in range(0, L, 128):
        pattern[n: n + 32, n: n + 32] = holes[n: n + 32, n: n + 32] if n % 256 else 1.0
        pattern[n: n + 32, (n + 512) % L: (n + 512) % L + 32] = 1.0
    return pattern


# tiles of one and of four wavefronts a strip; the remainder by ranges and gathered
@pytest.mark.parametrize("half,B,masked", [(0, 16, False), (40, 16, False), (40, 16, True), (100, 16, False), (230, 16, False), (40, 1, False),
                                           (230, 1, True)])
def test_infinities_stay_with_their_entries(half, B, masked):
    """An infinity or NaN of a row or column reaches the rows and columns it has an entry with and no other, also where a well-filled
    tile lacks the entry."""
    H, L = 2, 1024
    gen = torch.Generator(device="cuda").manual_seed(9 + half)
    pattern = _holed(L, half, gen)
    row, col = 128 + 11, 128 + 7
    heads = [torch.randn(B, H, L, 32, generator=gen, device="cuda") for _ in range(4)]
    cpp, handle, module = _module(B, H, L, masked)
    ones = torch.ones(B, L, device="cuda")
    core = _lib.core()

    def run(q, k, v, do):
        q, k, v = (t.requires_grad_() for t in (q, k, v))
        out, _ = module(q, k, v, ones, pattern)
        out.backward(do)
        assert core.spion_last_path(handle) == (3 if half else 2) and core.spion_debug_counter(handle, 3) == (B > 1)
        return out.detach(), q.grad, k.grad, v.grad

    clean = run(*(t.clone() for t in heads))

    def step(which, at, feature):
        """Which rows are finite.  They are those of the run without the infinity, to rounding."""
        inputs = [t.clone() for t in heads]
        inputs[which][..., at, feature] = float("nan" if which < 2 else "inf")  # (a logit of -inf is a probability of 0)
        finite = []
        for x, y in zip(run(*inputs), clean):
            ok = torch.isfinite(x).all(-1)
            # a few hundred terms of 2^-24 of a typical element each, in another order
            assert ((x - y).abs() <= 1e-5 * (y.abs() + y.pow(2).mean().sqrt()))[ok].all()
            finite.append(ok)
        return finite

    in_col, in_row, others = pattern[:, col] > 0, pattern[row] > 0, torch.arange(L, device="cuda") != row
    same = lambda finite, reached: torch.equal(finite, (~reached).expand_as(finite))
    for which in (1, 2):  # K, V: the rows that have the column
        out, dq, dk, dv = step(which, col, 3)
        reached = (pattern[in_col] > 0).any(0)  # dK and dV take {dS, P} of those rows
        assert same(out, in_col) and same(dq, in_col) and same(dk, reached)
        assert same(dv, reached if which == 1 else torch.zeros_like(reached))
    for which in (0, 3):  # Q, dO: the row itself and the columns that it has
        out, dq, dk, dv = step(which, row, 5)
        assert same(out, ~others if which == 0 else torch.zeros_like(others)) and same(dq, ~others)
        assert same(dk, in_row) and same(dv, in_row)
    cpp.destroy(handle)


def _scattered(L, gen, share=0.05):
    """A pattern without dense structure, a long row and an empty one."""
    pattern = (torch.rand(L, L, generator=gen, device="cuda") < share).float()
    pattern[17, ::2] = 1.0
    pattern[9] = 0.0
    return pattern


def _registered(handle, pattern):
    """The index of a pattern on file with a handle: (device tensors, number of entries)."""
    where, L = pattern.bool(), pattern.shape[0]
    off = torch.zeros(L + 1, dtype=torch.int32)
    off[1:] = where.sum(1).cumsum(0).cpu()
    col = where.nonzero()[:, 1].to(torch.int32).cpu()
    index = off.cuda(), col.cuda(), where.sum(1).to(torch.int32)
    nnz = int(off[-1])
    core = _lib.core()
    assert core.spion_register_pattern(handle, index[0].data_ptr(), index[1].data_ptr(), nnz, off.data_ptr(), col.data_ptr()) == 0
    return index, nnz


def test_scattered_patterns_and_capture():
    """A pattern without dense structure, without scratch (the element kernels) and with (the kernels by ranges): float64 agrees,
    and graphs of both give the eager bits, recorded before the handle has run anything."""
    B, H, L = 32, 2, 576
    gen = torch.Generator(device="cuda").manual_seed(3)
    pattern = _scattered(L, gen)
    q, k, v, do = (torch.randn(B, H, L, 32, generator=gen, device="cuda") for _ in range(4))
    where = pattern.bool()
    core = _lib.core()
    cpp, handle, _ = _module(B, H, L, False)
    (d_off, d_col, row_counts), nnz = _registered(handle, pattern)
    ds = torch.empty(B * H * nnz, device="cuda")
    out = torch.empty_like(q)
    p = torch.empty(B * H, nnz, device="cuda")
    grads = [torch.empty_like(q) for _ in range(3)]
    need = [core.spion_attn_scratch(handle, d_off.data_ptr(), d_col.data_ptr(), nnz, back) for back in (0, 1)]
    assert need[0] > 0 and need[1] >= B * H * nnz and core.spion_debug_counter(handle, 3) == 1
    scratch = torch.empty(max(need), device="cuda")

    def plain():
        at = (d_off.data_ptr(), d_col.data_ptr(), row_counts.data_ptr(), nnz)
        core.spion_attn_forward_rowmajor(handle, q.data_ptr(), k.data_ptr(), v.data_ptr(), None, p.data_ptr(), out.data_ptr(), *at)
        core.spion_attn_backward_rowmajor(handle, q.data_ptr(), k.data_ptr(), v.data_ptr(), p.data_ptr(), out.data_ptr(),
                                          do.data_ptr(), ds.data_ptr(), *(g.data_ptr() for g in grads), *at)

    def with_scratch():
        at = (d_off.data_ptr(), d_col.data_ptr(), nnz, H)
        core.spion_attn_forward_scratch(handle, q.data_ptr(), k.data_ptr(), v.data_ptr(), None, 0, p.data_ptr(), out.data_ptr(), *at,
                                        None, None, scratch.data_ptr(), need[0])
        core.spion_attn_backward_scratch(handle, q.data_ptr(), k.data_ptr(), v.data_ptr(), p.data_ptr(), out.data_ptr(), do.data_ptr(),
                                         *(g.data_ptr() for g in grads), *at, None, None, None, scratch.data_ptr(), need[1])

    def record(step):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            core.spion_set_stream(handle, torch.cuda.current_stream().cuda_stream)
            step()
        _lib.check_error("capture")
        return graph

    def results(run):
        for t in (out, p, *grads, scratch):
            t.fill_(float("nan"))
        run()
        torch.cuda.synchronize()
        return [t.clone() for t in (out, p, *grads)]

    steps = plain, with_scratch
    graphs = [record(step) for step in steps]
    core.spion_set_stream(handle, torch.cuda.current_stream().cuda_stream)
    eager = [results(step) for step in steps]
    _lib.check_error("steps")
    assert core.spion_last_path(handle) == 2
    assert not torch.equal(eager[0][0], eager[1][0])  # other kernels, other roundings
    for _ in range(3):
        for graph, want in zip(graphs, eager):
            assert all(torch.equal(x, y) for x, y in zip(results(graph.replay), want))
    at = lambda t: t[B // 2, 1][None]
    ref = _reference(at(q), at(k), at(v), at(do), pattern.double()[None], None)
    for got in eager:
        got = (got[1][(B // 2) * H + 1],) + tuple(at(got[i]) for i in (0, 2, 3, 4))
        for name, x, y in zip(("P", "out", "dQ", "dK", "dV"), got, (ref[0][0][where],) + ref[1:]):
            tol = 1e-5 * (y.abs() + y.pow(2).mean().sqrt())
            assert float(((x.double() - y).abs() / tol).max()) <= 1.0, name
    core.spion_set_stream(handle, 0)
    cpp.destroy(handle)


@pytest.mark.parametrize("kind", ["scattered", "window"])
@pytest.mark.parametrize("views", [False, True])
def test_calls_share_nothing_in_the_handle(kind, views):
    """Two steps of one module on two streams at a time: the bits of the same steps one after the other."""
    B, H, L = 32, 2, 1024
    gen = torch.Generator(device="cuda").manual_seed(4)
    pattern = _scattered(L, gen) if kind == "scattered" else _pattern(L, gen)
    shape = (B, L, H, 32) if views else (B, H, L, 32)
    make = lambda: torch.randn(*shape, generator=gen, device="cuda")
    inputs = [[make().transpose(1, 2) if views else make() for _ in range(4)] for _ in range(2)]
    ones = torch.ones(B, L, device="cuda")
    cpp, handle, module = _module(B, H, L, False)

    def step(which):
        q, k, v = (t.detach().requires_grad_() for t in inputs[which][:3])
        out, p = module(q, k, v, ones, pattern)
        out.backward(inputs[which][3])
        return out.detach(), p.detach(), q.grad, k.grad, v.grad

    want = [step(0), step(1)]
    assert _lib.core().spion_debug_counter(handle, 3) == 1
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    for s in streams:
        s.wait_stream(torch.cuda.current_stream())
    got = [[], []]
    for _ in range(4):
        for which, s in enumerate(streams):
            with torch.cuda.stream(s):
                got[which].append(step(which))
    torch.cuda.synchronize()
    for which in range(2):
        for results in got[which]:
            assert all(torch.equal(x, y) for x, y in zip(results, want[which]))
    cpp.destroy(handle)


@pytest.mark.parametrize("node", [True, False])
def test_no_memory_for_scratch(node, monkeypatch):
    """What fits without the scratch still runs: the element kernels, in P and dS."""
    B, H, L = 32, 2, 2048
    if not node:
        monkeypatch.setattr(_lib, "autograd_node", lambda: None)
    gen = torch.Generator(device="cuda").manual_seed(12)
    pattern = _scattered(L, gen)
    q, k, v, do = (torch.randn(B, H, L, 32, generator=gen, device="cuda") for _ in range(4))
    q, k, v = (t.requires_grad_() for t in (q, k, v))
    ones = torch.ones(B, L, device="cuda")
    cpp, handle, module = _module(B, H, L, False)
    core = _lib.core()

    def step(limit):
        """Forward and backward, with no more than 1.5 times P and the tensors beside the inputs in either."""
        q.grad = k.grad = v.grad = None
        with torch.no_grad():
            p_bytes = 4 * B * H * int(pattern.sum())
        for part in ("forward", "backward"):
            torch.cuda.synchronize()
            torch.cuda.empty_cache()
            if limit:
                room = torch.cuda.memory_reserved() + 1.5 * p_bytes + 4 * q.numel() * (1 if part == "forward" else 3)
                torch.cuda.set_per_process_memory_fraction(room / torch.cuda.get_device_properties(0).total_memory)
            try:
                if part == "forward":
                    out, p = module(q, k, v, ones, pattern)
                else:
                    out.backward(do)
            finally:
                torch.cuda.set_per_process_memory_fraction(1.0)
        return out.detach(), p.detach(), q.grad, k.grad, v.grad

    want = step(False)
    assert core.spion_debug_counter(handle, 3) == 1
    got = step(True)
    assert not torch.equal(got[0], want[0])  # other kernels, other roundings
    for x, y in zip(got, want):
        assert ((x - y).abs() <= 1e-5 * (y.abs() + y.pow(2).mean().sqrt())).all()
    cpp.destroy(handle)


# long patterns of few entries, few heads: gathered, whether mostly tiles or not; an empty remainder
@pytest.mark.parametrize("B,L,kind", [(4, 4096, "scattered"), (1, 8192, "scattered"), (4, 4096, "window"), (64, 1024, "tiles")])
def test_patterns_that_are_gathered(B, L, kind):
    gen = torch.Generator(device="cuda").manual_seed(6)
    i = torch.arange(L, device="cuda")
    if kind == "tiles":  # whole tiles but for one entry of each
        pattern = ((i[:, None] // 32 - i[None, :] // 32).abs() <= 1).float()
        pattern[::32, ::32] = 0.0
    else:
        pattern = (torch.rand(L, L, generator=gen, device="cuda") < 16 / L).float()
        if kind == "window":
            pattern[(i[:, None] - i[None, :]).abs() <= 40] = 1.0
    q, k, v, do = (torch.randn(B, 1, L, 32, generator=gen, device="cuda") for _ in range(4))
    q, k, v = (t.requires_grad_() for t in (q, k, v))
    cpp, handle, module = _module(B, 1, L, False)
    out, p = module(q, k, v, torch.ones(B, L, device="cuda"), pattern)
    out.backward(do)
    core = _lib.core()
    assert core.spion_debug_counter(handle, 3) == 0 and core.spion_last_path(handle) == (2 if kind == "scattered" else 3)
    at = lambda t: t.detach()[B - 1]
    ref = _reference(at(q), at(k), at(v), at(do), pattern.double()[None], None)
    got = (p.detach().reshape(B, -1)[B - 1],) + tuple(at(t) for t in (out, q.grad, k.grad, v.grad))
    for name, x, y in zip(("P", "out", "dQ", "dK", "dV"), got, (ref[0][0][pattern.bool()],) + ref[1:]):
        tol = 1e-5 * (y.abs() + y.pow(2).mean().sqrt())
        assert float(((x.double() - y).abs() / tol).max()) <= 1.0, name
    cpp.destroy(handle)
