"""Performance cases: the work a program that uses spion_amd has it do, through the public entry points.

A case is a dict of plain values:

  path       sparse       ``CUDABlockAttention``: block mask, fp32, returns the probabilities
             sparse_mask  ``CUDABlockMaskAttention``: block mask and key padding, fp32
             element      ``CUDABlockMaskAttention`` with block size 1: a +-64 window and random columns in every row
             bf16         ``BlockAttentionBF16``: block mask (band, one global block row and column, random blocks)
             dense        ``CUDAAttention``: the dense phase, full probability maps, fp32
             dense_mask   ``CUDAMaskAttention``: the same with key padding
             layer        ``Attention`` in its sparse phase: projections, sparse core, output projection
             discovery    ``generate_pattern_conv_ff``: score maps of all layers -> block masks
  direction  train: forward and backward; infer: forward without gradients (dense: with the mean score map, as the
             evaluation ahead of pattern discovery runs it)
  batch, heads, length, head_dim, block   the config a module is built with
  density    share of the blocks (element: of the columns of a row) that the mask keeps
  masked     layer, bf16: with key padding

``listed`` holds the fixed cases, ``draw`` gives others of the same ranges.
"""
import math
import weakref

import torch

import spion_amd
from spion_amd import _lib, workloads


def _case(name, path, direction, batch, heads, length, head_dim, block, density, masked=False):
    return {"name": name, "path": path, "direction": direction, "batch": batch, "heads": heads, "length": length,
            "head_dim": head_dim, "block": block, "density": density, "masked": masked}


def listed():
    return [
        # Evaluation of single samples with saved masks: one layer of the padded-text task, batch 1.  Latency.
        _case("layer_infer_single", "layer", "infer", 1, 2, 2048, 32, 64, 0.06, masked=True),
        # A training step of one attention core at L = 1024 with a small batch: kernels of microseconds, host and
        # launches count.
        _case("sparse_train_short", "sparse", "train", 8, 2, 1024, 32, 32, 0.136),
        # The same core at the batch size the image task trains with.
        _case("sparse_train_batch", "sparse", "train", 256, 2, 1024, 32, 32, 0.136),
        # The long-sequence training step: L = 4096, a tenth of the blocks kept.
        _case("sparse_train_long", "sparse", "train", 32, 2, 4096, 32, 32, 0.10),
        # Text tasks: key padding, 64x64 blocks, the density a high quantile leaves.
        _case("sparse_mask_train_text", "sparse_mask", "train", 32, 2, 2048, 32, 64, 0.06),
        # Wider heads and sizes off the powers of two: 4000 tokens, three samples of eight heads of 64 features.
        _case("sparse_train_wide_ragged", "sparse", "train", 3, 8, 4000, 64, 32, 0.08),
        # Element-sparse attention with key padding: a local window and random columns, 5 % of each row.
        _case("element_train_padded", "element", "train", 32, 2, 4096, 32, 1, 0.05),
        # The whole attention layer in training: fused projections, heads read in place, output projection.
        _case("layer_train", "layer", "train", 64, 2, 1024, 32, 32, 0.12),
        # Scale-up training step in bf16: 16384 tokens, band + global row and column + random blocks.
        _case("bf16_train_scale_up", "bf16", "train", 4, 8, 16384, 64, 64, 0.037),
        # Serving in bf16 with padding: forward only, moderate batch.
        _case("bf16_infer_padded", "bf16", "infer", 4, 8, 4096, 64, 64, 0.08, masked=True),
        # The dense phase that precedes discovery: full maps, forward and backward.
        _case("dense_train", "dense", "train", 64, 2, 1024, 32, 32, 1.0),
        # Pattern discovery for a model of four layers at L = 2048.
        _case("discovery_four_layers", "discovery", "infer", 4, 1, 2048, 32, 32, 0.10),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


# (lengths, batch * heads, densities) a path is drawn from; both ends are in use
_RANGES = {
    "sparse": ((512, 8192), (2, 512), (0.03, 0.20)),
    "sparse_mask": ((512, 8192), (2, 512), (0.03, 0.20)),
    "element": ((1024, 4096), (16, 64), (0.04, 0.08)),
    "bf16": ((1024, 16384), (4, 128), (0.02, 0.15)),
    "dense": ((256, 2048), (4, 256), (1.0, 1.0)),
    "dense_mask": ((256, 2048), (4, 256), (1.0, 1.0)),
    "layer": ((512, 4096), (2, 256), (0.03, 0.20)),
    "discovery": ((1024, 4096), (1, 6), (0.02, 0.10)),
}


def draw(rng):
    most_bytes = max(work(c)["bytes"] for c in listed())
    most_flops = {fp: max(work(c)["flops"] for c in listed() if (c["path"] == "bf16") == fp) for fp in (False, True)}
    while True:
        path = rng.choice(sorted(_RANGES))
        lengths, heads_total, densities = _RANGES[path]
        direction = "infer" if path == "discovery" or rng.random() < 0.3 else "train"
        block = 1 if path == "element" else rng.choice((32, 64))
        head_dim = 32 if path in ("element", "discovery") or rng.random() < 0.6 else 64
        length = int(_log_uniform(rng, *lengths))
        # the kernels' unit is 32 rows; block masks need whole blocks
        length = max(1, round(length / max(block, 32))) * max(block, 32)
        heads = 1 if path == "discovery" else rng.choice((1, 2, 2, 3, 4, 8))
        batch = max(1, round(_log_uniform(rng, *heads_total) / heads))
        masked = path in ("layer", "bf16") and rng.random() < 0.5
        c = _case(None, path, direction, batch, heads, length, head_dim, block,
                  round(_log_uniform(rng, *densities), 4), masked)
        del c["name"]
        w = work(c)
        if w["bytes"] <= most_bytes and w["flops"] <= most_flops[path == "bf16"]:
            return c


def _is_masked(c):
    return c["path"] in ("sparse_mask", "element", "dense_mask") or c["masked"]


def _entries(c):
    """Entries of the pattern per head."""
    L = c["length"]
    if c["path"] in ("dense", "dense_mask"):
        return L * L
    if c["path"] == "element":
        return L * max(2, round(c["density"] * L))
    nb = L // c["block"]
    if c["path"] == "bf16":
        return int(_block_mask(c, 0).sum()) * c["block"] ** 2
    return max(round(c["density"] * nb * nb), 3 * nb - 2) * c["block"] ** 2


def _block_mask(c, seed):
    """Kept blocks: a band of three and random others up to the density (never fewer than the band); the bf16 cases
    add one global block row and column."""
    nb = c["length"] // c["block"]
    if c["path"] == "bf16":
        rest = max(0.0, c["density"] * nb - 7.0) / nb  # what a band of five and the global blocks leave
        mat = workloads.band_random_block_mask(nb, 2, extra_frac=rest, seed=seed)
        mat[0, :] = 1.0
        mat[:, 0] = 1.0
        return mat
    return workloads.band_random_block_mask(nb, 1, density=c["density"], seed=seed)


def work(c):
    """Bytes and operations a pass cannot do without: every input read once, every returned tensor written once (the
    probabilities where they are returned); two products per entry forward, four more backward."""
    B, H, L, d = c["batch"], c["heads"], c["length"], c["head_dim"]
    NB = B * H
    if c["path"] == "discovery":
        nb = L // c["block"]
        return {"bytes": 4.0 * B * (L * L + 4 * nb * nb), "flops": 2.0 * B * L * L}
    train = c["direction"] == "train"
    n = _entries(c)
    size = 2.0 if c["path"] == "bf16" else 4.0
    tensors = size * L * d * NB * (8 if train else 4)
    returned = 4.0 * n * NB if c["path"] in ("sparse", "dense", "dense_mask") or (
        c["path"] == "layer" and not c["masked"]) else 0.0
    index = 4.0 * (L // c["block"]) ** 2 if c["path"] not in ("dense", "dense_mask") else 0.0
    flops = (12.0 if train else 4.0) * n * d * NB
    nbytes = tensors + returned + index + (4.0 * B * L if _is_masked(c) else 0.0)
    if c["path"] in ("dense", "dense_mask") and not train:
        nbytes += 4.0 * L * L  # the mean score map
    if c["path"] == "layer":
        dim = H * d
        # X and Y (and their gradients) instead of Q, K, V, O; weights; four projections of dim x dim
        nbytes = size * B * L * dim * (4 if train else 2) + returned + index + 16.0 * dim * dim * (2 if train else 1)
        flops += (3.0 if train else 1.0) * 4 * 2.0 * B * L * dim * dim
    return {"bytes": nbytes, "flops": flops}


def tolerance(c):
    if c["path"] == "discovery":
        return "exact"  # the masks are integers by contract
    if c["path"] == "bf16":
        return {"rel": 1e-2}
    return {"rel": 1e-5}


class _State:
    """What a program keeps between passes.  The library's handles are freed with it."""

    def __init__(self, case, **kept):
        self.case = case
        self.__dict__.update(kept)


def _owned(module, destroy):
    weakref.finalize(module, destroy, module.attn_handle)
    return module


def _normal(gen, *shape, scale=1.0, dtype=torch.float32):
    return (torch.randn(*shape, generator=gen, device="cuda") * scale).to(dtype)


def _element_mask(c, gen):
    """[L, L] 0/1: columns within 64 of the row and random others, the same number in every row."""
    L = c["length"]
    per_row = max(2, round(c["density"] * L))
    score = torch.rand(L, L, generator=gen, device="cuda")
    i = torch.arange(L, device="cuda")
    score += 1.0 * ((i[:, None] - i[None, :]).abs() <= min(64, per_row // 3))
    mat = torch.zeros(L, L, device="cuda")
    mat.scatter_(1, score.topk(per_row, dim=1).indices, 1.0)
    return mat


def _key_mask(c, gen):
    B, L = c["batch"], c["length"]
    if not _is_masked(c):
        return torch.ones(B, L, device="cuda")
    valid = torch.randint(L // 2, L + 1, (B, 1), generator=gen, device="cuda")
    return (torch.arange(L, device="cuda")[None, :] < valid).to(torch.float32)


def _score_maps(c, gen):
    """Averaged attention maps as a trained dense phase leaves them: softmax rows with a diagonal band."""
    L, d = c["length"], c["head_dim"]
    i = torch.arange(L, device="cuda")
    maps = []
    for layer in range(c["batch"]):
        q, k = _normal(gen, L, d), _normal(gen, L, d)
        a = torch.softmax(q @ k.t() / math.sqrt(d), dim=-1)
        band = (i[None, :] - i[:, None] - 17 * layer).abs() <= 8 + 4 * layer
        maps.append(a + 3.0 * a.std() * band)
    return maps


def prepare(case, seed):
    c = dict(case)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    B, H, L, d, path = c["batch"], c["heads"], c["length"], c["head_dim"], c["path"]
    if path == "discovery":
        config = {"block_size": c["block"], "max_seq_len": L, "num_layers": B, "threshold": 1.0 - c["density"]}
        return _State(c, maps=_score_maps(c, gen), config=config)
    train = c["direction"] == "train"
    config = {"head_dim": d, "num_head": H, "max_seq_len": L, "batch_size": B, "block_size": c["block"],
              "transformer_dim": H * d, "attention_dropout": 0.0, "task": "lra-text" if c["masked"] else "lra-image"}
    mask = _key_mask(c, gen)
    mat = None
    if path == "element":
        mat = _element_mask(c, gen)
    elif path not in ("dense", "dense_mask"):
        mat = torch.from_numpy(_block_mask(c, seed)).to("cuda")

    if path == "layer":
        with torch.random.fork_rng(devices=[0]):
            torch.manual_seed(seed)
            layer = spion_amd.Attention(config, inference=True).to("cuda")
        layer.reconstruct_for_blocksparse(config)
        lib = _lib.core()
        _owned(layer.block_attn, lib.spion_blockmask_destroy if c["masked"] else lib.spion_block_destroy)
        masks = mat[None, None]
        spion_amd.attach_mask_sidecars([layer], masks, config)
        x = _normal(gen, B, L, H * d).requires_grad_(train)
        dy = _normal(gen, B, L, H * d)
        return _State(c, layer=layer, x=x, dy=dy, mask=mask, mat=masks[0][0])

    dtype, scale = (torch.bfloat16, 1.0 / 8.0) if path == "bf16" else (torch.float32, 1.0)
    if path == "bf16":
        module = _owned(spion_amd.BlockAttentionBF16(config, key_mask=c["masked"]), _lib.core().spion_block_bf16_destroy)
    else:
        load, cls, sizes = {
            "sparse": ("_blockcuda_compile_module", spion_amd.CUDABlockAttention, (d, L, B * H, c["block"])),
            "sparse_mask": ("_blockcuda_mask_compile_module", spion_amd.CUDABlockMaskAttention, (d, L, B * H, c["block"])),
            "element": ("_blockcuda_mask_compile_module", spion_amd.CUDABlockMaskAttention, (d, L, B * H, c["block"])),
            "dense": ("_cuda_compile_module", spion_amd.CUDAAttention, (d, L, B * H)),
            "dense_mask": ("_cuda_mask_compile_module", spion_amd.CUDAMaskAttention, (d, L, B * H)),
        }[path]
        cpp = getattr(spion_amd.Attention, load)()
        module = _owned(cls(config, cpp, cpp.init(*sizes)), cpp.destroy)
        if path in ("dense", "dense_mask") and not train:
            module.emit_score_map = True
    q, k, v = (_normal(gen, B, H, L, d, scale=scale, dtype=dtype).requires_grad_(train) for _ in range(3))
    do = _normal(gen, B, H, L, d, dtype=dtype)
    return _State(c, module=module, q=q, k=k, v=v, do=do, mask=mask, mat=mat)


def _attend(s):
    if s.mat is None:
        return s.module(s.q, s.k, s.v, s.mask)
    return s.module(s.q, s.k, s.v, s.mask, s.mat)


def run(s):
    c = s.case
    if c["path"] == "discovery":
        return spion_amd.generate_pattern_conv_ff(s.maps, s.config)
    if c["path"] == "layer":
        if c["direction"] == "infer":
            with torch.no_grad():
                return s.layer(s.x, s.mask, s.mat)
        s.x.grad = None
        s.layer.zero_grad(set_to_none=True)
        y, attn = s.layer(s.x, s.mask, s.mat)
        y.backward(s.dy)
        return [y, attn, s.x.grad] + [p.grad for p in s.layer.parameters()]
    if c["direction"] == "infer":
        with torch.no_grad():
            out, attn = _attend(s)
        return [out, attn, s.module.score_map] if s.mat is None else [out, attn]
    s.q.grad = s.k.grad = s.v.grad = None
    out, attn = _attend(s)
    out.backward(s.do)
    return [out, attn, s.q.grad, s.k.grad, s.v.grad]
