"""The work a user of this framework has it do, as measurable cases.

A case is a dict of plain values.  ``kind`` names the entry point it goes through:

* ``restore`` -- ``restore_kernels.reconstruct`` of one or more layers: archived 8-bit (rows or
  channel_tiles.v1 pictures), float or dense sources into native K / V cache slots, eagerly or as
  replays of a captured HIP graph (a serving loop's layer restores);
* ``tile`` -- ``factorization.project_onto_basis`` and ``node_packets.quantize_device`` of one matrix
  (archiving one matrix on a basis at hand);
* ``gram`` -- ``fit_kernels.gram`` of a batch of matrices;
* ``plan`` -- ``GramPlanner.plan`` of a chunk's matrices (rank and basis decisions);
* ``finalize`` -- ``node_packets.finalize_tiles`` of a chunk's matrices on planned rows.

``prepare`` makes inputs of the distributions the path meets: orthonormal bases, coefficients
whose column scale decays like singular values do (``k ** -0.8``) and whose 8-bit codes cover
+-4 standard deviations, and sources of a decaying spectrum plus noise.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from reelcache_amd import factorization, fit_kernels
from reelcache_amd import gpu_fitting, rank_method
from reelcache_amd import node_packets as npk
from reelcache_amd import restore_kernels as rk
from reelcache_amd.quantize import covering_affine, video_layout
from reelcache_amd.types import CodecSpec, MatrixKey, ModelIdentity, TensorContext, energy_targets

DEVICE = "cuda:0"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
SIZES = {"bf16": 2, "fp16": 2, "fp32": 4}

# Defaults of a restore case: one layer, K and V of every chunk, uint8 rows, fp16x2 into bf16.
RESTORE = {"kind": "restore", "source": "codes", "layers": 1, "graph": False, "chunks": 1, "frames": 3, "height": 30,
           "width": 52, "heads": 12, "head_dim": 128, "rank_k": 128, "rank_v": 192, "rank_low": 0, "layout": "BTHD",
           "rope": "separable", "precision": "auto", "basis": "bf16", "out": "bf16", "coefficients": "fp32"}
FIT = {"matrices": 60, "frames": 3, "height": 30, "width": 52, "channels": 1536, "dtype": "bf16"}


def listed():
    return [
        # The smallest call: the K and V of one short chunk of one layer at low rank (a rewound tip).
        dict(RESTORE, name="restore_short_chunk", frames=1, height=15, width=26, rank_k=32, rank_v=32),
        # One layer of a whole CausVid history: seven chunks of K (Wan RoPE) and V in one call.
        dict(RESTORE, name="restore_history_layer", chunks=7),
        # Four such layers as a serving loop replays them from a captured graph.
        dict(RESTORE, name="restore_history_graph", chunks=7, layers=4, graph=True),
        # The same history layer from decoded pictures (the stored form of an archive).
        dict(RESTORE, name="restore_history_pictures", chunks=7, source="pictures"),
        # A LongCat-shaped layer: [B, H, T, D] caches, 32 heads, ranks 256 to 512, no RoPE.
        dict(RESTORE, name="restore_wide_layer", chunks=8, heads=32, rank_k=512, rank_v=512, rank_low=256,
             layout="BHTD", rope="none"),
        # Two chunks of that shape from decoded pictures.
        dict(RESTORE, name="restore_wide_pictures", chunks=2, source="pictures", heads=32, rank_k=512, rank_v=512,
             rank_low=256, layout="BHTD", rope="none"),
        # Odd sizes: code rows of 75 bytes, heads of 80 channels, dense RoPE, an fp16 cache.
        dict(RESTORE, name="restore_ragged", chunks=3, frames=2, height=17, width=29, heads=5, head_dim=80, rank_k=75,
             rank_v=75, layout="BHTD", rope="dense", basis="fp16", out="fp16"),
        # Uncompressed chunks (the recent part of a history) rotated and stored into the caches.
        dict(RESTORE, name="restore_dense_slots", chunks=3, source="dense", coefficients="bf16"),
        # One matrix archived on an inherited basis: projection, residual guard, codes.
        dict(FIT, name="archive_one_tile", kind="tile", matrices=1, rank=96),
        # The Gram matrices of one chunk (30 layers of K and V).
        dict(FIT, name="gram_chunk", kind="gram"),
        # Rank and basis decisions of one chunk.
        dict(FIT, name="plan_chunk", kind="plan"),
        # Stored measurement and codes of one chunk at ranks 32 to 128.
        dict(FIT, name="finalize_chunk", kind="finalize", rank=128),
    ]


def _span(rng, low, high):
    """An integer of [low, high], even over the logarithm."""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    kind = rng.choice(["codes", "codes", "codes", "pictures", "pictures", "float", "dense", "tile", "gram", "plan",
                       "finalize"])
    grid = {"frames": rng.randint(1, 3), "height": rng.randint(9, 30), "width": rng.randint(13, 52)}
    if kind in ("tile", "gram", "plan", "finalize"):
        case = dict(FIT, kind=kind, **grid, channels=8 * rng.randint(40, 192), dtype=rng.choice(["bf16", "bf16", "fp16", "fp32"]),
                    matrices=1 if kind == "tile" else _span(rng, 2, 60))
        if kind in ("tile", "finalize"):
            case["rank"] = min(16 * rng.randint(1, 8), grid["frames"] * grid["height"] * grid["width"])
        if case["dtype"] == "fp32":
            case["matrices"] = min(case["matrices"], 12)
        return case
    case = dict(RESTORE, source=kind, **grid, chunks=rng.randint(1, 7), heads=_span(rng, 2, 32),
                head_dim=rng.choice([64, 80, 96, 128, 128]), layout=rng.choice(["BTHD", "THD", "BHTD"]),
                rope=rng.choice(["separable", "separable", "dense", "none"]), basis=rng.choice(["bf16", "fp16"]),
                out=rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"]))
    if kind == "dense":
        return dict(case, coefficients=rng.choice(["bf16", "fp16", "fp32"]))
    most = min(512, case["frames"] * case["height"] * case["width"], case["heads"] * case["head_dim"])
    odd = kind == "codes" and rng.random() < 0.25  # rows that are not 16-byte aligned
    for name in ("rank_k", "rank_v"):
        rank = _span(rng, 8, most)
        case[name] = rank if odd else min(most, -(-rank // 16) * 16)
    case["precision"] = rng.choice(["auto", "auto", "auto", "fp16", "bf16", "fp32"])
    case["coefficients"] = rng.choice(["fp32", "fp32", "fp16"])
    if case["precision"] == "fp32" or kind == "float":
        case["chunks"] = min(case["chunks"], 3)
    return case


# ---------------------------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------------------------


def _tokens(case):
    return case["frames"] * case["height"] * case["width"]


def _rank(case, target, chunk):
    """Chunk ``chunk``'s rank: the target's, or spread over the 32-grid from ``rank_low`` to it."""
    rank = case["rank_k"] if target == 0 else case["rank_v"]
    if not case["rank_low"]:
        return rank
    steps = (rank - case["rank_low"]) // 32 + 1
    return case["rank_low"] + 32 * ((5 * chunk + 3 * target + steps - 1) % steps)


def _generator(seed, salt=0):
    return torch.Generator(device=DEVICE).manual_seed(1000003 * (seed % (1 << 40)) + salt)


def _orthonormal(rows, channels, generator, dtype):
    q = torch.linalg.qr(torch.randn(channels, rows, device=DEVICE, generator=generator)).Q
    return q.T.contiguous().to(dtype)


def _decay(rank):
    return torch.arange(1, rank + 1, dtype=torch.float64) ** -0.8


def _affine(rank, rng):
    """Covering affine of columns spread over +-4 standard deviations around a small mean."""
    sigma = 30.0 * _decay(rank).numpy()
    middle = rng.uniform(-0.5, 0.5, size=rank) * sigma
    affine = covering_affine((middle - 4 * sigma).astype(np.float32), (middle + 4 * sigma).astype(np.float32))
    return affine[0].copy(), affine[1].copy()


def _codes(tokens, rank, generator):
    return (torch.randn(tokens, rank, device=DEVICE, generator=generator) * 32 + 127.5).round().clamp(0, 255).to(torch.uint8)


def _table(case, tokens):
    pairs = case["head_dim"] // 2
    if case["rope"] == "none":
        return None
    if case["rope"] == "dense":
        angles = torch.outer(torch.arange(tokens + 8, dtype=torch.float64),
                             10000.0 ** (-torch.arange(pairs, dtype=torch.float64) / pairs))
        return rk.RopeTable.from_cos_sin(angles.cos().float(), angles.sin().float())
    sixth = case["head_dim"] // 6
    parts = []
    for dim in (case["head_dim"] - 4 * sixth, 2 * sixth, 2 * sixth):
        inverse = 1.0 / 10000.0 ** (torch.arange(0, dim, 2, dtype=torch.float64) / dim)
        angles = torch.outer(torch.arange(64, dtype=torch.float64), inverse)
        parts.append(torch.polar(torch.ones_like(angles), angles))
    return rk.RopeTable.from_complex(torch.cat(parts, dim=1))


def _rope_rows(case, chunk):
    return (case["frames"] * chunk, 0, 0) if case["rope"] == "separable" else 3


def _restore_layers(case, seed):
    """Per layer and target the shared basis and per chunk (rank, values, scale, offset): the inputs
    of a restore case, the same for the kernels and for the 64-bit values."""
    tokens, channels = _tokens(case), case["heads"] * case["head_dim"]
    rng = np.random.default_rng(seed % (1 << 32))
    generator = _generator(seed)
    layers = []
    for _ in range(case["layers"]):
        targets = []
        for target in (0, 1):
            ranks = [_rank(case, target, chunk) for chunk in range(case["chunks"])]
            if case["source"] == "dense":
                chunks = [(None, torch.randn(tokens, channels, device=DEVICE, generator=generator).to(
                    DTYPES[case["coefficients"]]), None, None) for _ in ranks]
                targets.append((None, chunks))
                continue
            basis = _orthonormal(max(ranks), channels, generator, DTYPES[case["basis"]])
            chunks = []
            for rank in ranks:
                if case["source"] == "float":
                    scale = 30.0 * _decay(rank).to(device=DEVICE, dtype=torch.float32)
                    values = (torch.randn(tokens, rank, device=DEVICE, generator=generator) * scale).to(
                        DTYPES[case["coefficients"]])
                    chunks.append((rank, values, None, None))
                else:
                    chunks.append((rank, _codes(tokens, rank, generator), *_affine(rank, rng)))
            targets.append((basis, chunks))
        layers.append(targets)
    return layers


def _source(case, rank, values, scale, offset):
    if case["source"] == "dense":
        return rk.DenseSource(values)
    if case["source"] == "float":
        return rk.CoefficientSource(values)
    if case["source"] == "codes":
        return rk.CoefficientSource(values, scale, offset)
    frames = case["frames"]
    video = video_layout(frames, case["height"], case["width"], rank, "yuv444p")
    canvases = npk.mosaic_device(values, video)
    indices = [[segment * frames + frame for frame in range(frames)] for segment in range(video["segments"])]
    return rk.PictureSource.from_canvases(canvases, video, indices, (0, 0), scale, offset)


def _prepare_restore(case, seed):
    tokens = _tokens(case)
    history = case["chunks"] * tokens
    heads, dim = case["heads"], case["head_dim"]
    shape = {"BTHD": (1, history, heads, dim), "THD": (history, heads, dim), "BHTD": (1, heads, history, dim)}[case["layout"]]
    table = _table(case, tokens)
    if table is not None:
        table.kernel_tables(torch.device(DEVICE))
    caches, calls = [], []
    grid = (case["frames"], case["height"], case["width"])
    for targets in _restore_layers(case, seed):
        jobs = []
        for target, (basis, chunks) in enumerate(targets):
            cache = torch.zeros(shape, dtype=DTYPES[case["out"]], device=DEVICE)
            caches.append(cache)
            for chunk, (rank, values, scale, offset) in enumerate(chunks):
                rope = None if target or table is None else rk.RopePositions(table, _rope_rows(case, chunk))
                view = rk.NativeView(cache, case["layout"], token_offset=chunk * tokens)
                jobs.append(rk.ReconstructionJob(_source(case, rank, values, scale, offset), view, grid, basis, rank, rope))
        calls.append(jobs)
    state = {"case": case, "caches": caches, "calls": calls}
    if case["graph"]:
        device = torch.device(DEVICE)
        for jobs in calls:
            rk.reconstruct(jobs, precision=case["precision"]).release()
        rk.reserve_capture_staging(len(calls) * (64 << 10))
        state["graph"] = graph = torch.cuda.CUDAGraph()
        stream = torch.cuda.Stream(device)
        stream.wait_stream(torch.cuda.current_stream(device))
        with torch.cuda.graph(graph, stream=stream):
            state["handles"] = [rk.reconstruct(jobs, precision=case["precision"], stream=stream) for jobs in calls]
        for cache in caches:
            cache.zero_()
    return state


def _run_restore(state):
    case = state["case"]
    if case["graph"]:
        state["graph"].replay()
    else:
        # The handles keep the inputs until the device is done; the next pass replaces them.
        state["handles"] = [rk.reconstruct(jobs, precision=case["precision"]) for jobs in state["calls"]]
    return state["caches"]


def _sources(case, seed):
    """The chunk's matrices: a decaying spectrum (sigma_i = i ** -0.9, random directions) plus noise."""
    tokens, channels = _tokens(case), case["channels"]
    generator = _generator(seed, 1)
    inner = min(256, tokens, channels)
    sigma = torch.arange(1, inner + 1, dtype=torch.float32, device=DEVICE) ** -0.9
    matrices = []
    for _ in range(case["matrices"]):
        left = torch.randn(tokens, inner, device=DEVICE, generator=generator) * sigma
        right = torch.randn(inner, channels, device=DEVICE, generator=generator) / math.sqrt(channels)
        noise = torch.randn(tokens, channels, device=DEVICE, generator=generator) * (2e-2 / math.sqrt(channels))
        matrices.append((left @ right + noise).to(DTYPES[case["dtype"]]))
    return matrices


def _contexts(case):
    layers = -(-case["matrices"] // 2)
    name = {"bf16": "bfloat16", "fp16": "float16", "fp32": "float32"}[case["dtype"]]
    model = ModelIdentity("causvid-synthetic", "c" * 64, layers, case["channels"], "THD", name)
    grid = (case["frames"], case["height"], case["width"])
    keys = [MatrixKey(index // 2, "KV"[index % 2]) for index in range(case["matrices"])]
    return {key: TensorContext(model, key, 0, *grid, "pre_rope" if key.target == "K" else "none") for key in keys}


def _ranks(case):
    """Planned ranks of a chunk: the bucket grid up to the case's rank, in turn."""
    step = 32 if case["rank"] >= 32 else 16
    count = max(1, case["rank"] // step)
    return [min(case["rank"], step * (1 + (5 * index) % count)) for index in range(case["matrices"])]


def _bases(case, matrices, seed):
    """FP16 rows spanning each matrix's leading directions (one subspace step of a random block)."""
    generator = _generator(seed, 2)
    rows = []
    for matrix, rank in zip(matrices, _ranks(case)):
        x = matrix.float()
        block = x.T @ (x @ torch.randn(case["channels"], rank, device=DEVICE, generator=generator))
        rows.append(torch.linalg.qr(block).Q.T.contiguous().to(torch.float16))
    return rows


def prepare(case, seed):
    if case["kind"] == "restore":
        return _prepare_restore(case, seed)
    state = {"case": case, "matrices": _sources(case, seed)}
    if case["kind"] == "tile":
        generator = _generator(seed, 2)
        state["basis"] = _orthonormal(case["rank"], case["channels"], generator, torch.float16)
        state["spec"] = CodecSpec("svd_hevc", case["rank"])
    elif case["kind"] == "plan":
        contexts = _contexts(case)
        keys = list(contexts)
        config = rank_method.RankMethodConfig(energy_targets("causvid"), CodecSpec("svd_hevc", 1))
        label, solver = gpu_fitting.select_eigh_solver("auto")
        state.update(planner=rank_method.GramPlanner(config, device=torch.device(DEVICE), eigh=solver, eigh_label=label),
                     contexts=contexts, sources=dict(zip(keys, state["matrices"])),
                     bindings={key: rank_method.ActiveBasisBinding() for key in keys},
                     parents={key: None for key in keys}, ids={key: str(key) for key in keys})
    elif case["kind"] == "finalize":
        contexts = _contexts(case)
        state["items"] = [npk.FinalizeItem(matrix, rows, context, CodecSpec("svd_hevc", int(rows.shape[0])), key, 0.5, True,
                                           rows.cpu())
                          for (key, context), matrix, rows in zip(contexts.items(), state["matrices"],
                                                                  _bases(case, state["matrices"], seed))]
    return state


# ---------------------------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------------------------


def run(state):
    kind = state["case"]["kind"]
    if kind == "restore":
        return _run_restore(state)
    if kind == "gram":
        return fit_kernels.gram(state["matrices"])
    if kind == "tile":
        projection = factorization.project_onto_basis(state["matrices"][0], state["basis"])
        pixels, affine, _ = npk.quantize_device(projection.coefficients, state["spec"])
        return {"coefficients": projection.coefficients, "codes": pixels, "affine": np.asarray(affine, dtype=np.float32),
                "residual": projection.relative_residual, "norm": projection.source_norm}
    if kind == "plan":
        plan = state["planner"].plan(state["sources"], state["contexts"], state["bindings"], state["parents"],
                                     chunk_id="chunk", source_ids=state["ids"])
        plans = [plan.plans[key] for key in state["sources"]]
        return {"rows": torch.cat([p.new_rows for p in plans]), "ranks": np.array([p.rank_view for p in plans]),
                "energies": np.array([p.decision_energy for p in plans])}
    results = npk.finalize_tiles(state["items"], tile_rows=1024)
    tiles = [tile for tile, _ in results]
    return {"codes": torch.cat([pixels.reshape(-1) for _, pixels in results]),
            "affine": np.concatenate([np.frombuffer(tile.affine, dtype="<f4") for tile in tiles]),
            "stored": np.array([tile.stored_energy for tile in tiles]),
            "span": np.array([tile.ideal_energy for tile in tiles]),
            "source": np.array([tile.source_energy for tile in tiles])}


# ---------------------------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------------------------


def work(case):
    tokens = _tokens(case)
    if case["kind"] == "restore":
        channels = case["heads"] * case["head_dim"]
        nbytes = flops = 0
        for target in (0, 1):
            ranks = [_rank(case, target, chunk) for chunk in range(case["chunks"])]
            nbytes += len(ranks) * tokens * channels * SIZES[case["out"]]
            if case["source"] == "dense":
                nbytes += len(ranks) * tokens * channels * SIZES[case["coefficients"]]
                continue
            size = SIZES[case["coefficients"]] if case["source"] == "float" else 1
            nbytes += sum(tokens * rank * size + 8 * rank for rank in ranks) + max(ranks) * channels * 2
            flops += sum(2 * tokens * channels * rank for rank in ranks)
        return {"bytes": case["layers"] * nbytes, "flops": case["layers"] * flops}
    channels, count = case["channels"], case["matrices"]
    source = tokens * channels * SIZES[case["dtype"]]
    if case["kind"] == "gram":  # each product of two columns once
        return {"bytes": count * (source + 4 * channels * channels), "flops": count * tokens * channels * (channels + 1)}
    if case["kind"] == "plan":
        # One Gram and the power steps of a 96-column block, then one measurement of the chosen rows.
        width = min(96, channels, tokens)
        return {"bytes": count * source, "flops": count * (tokens * channels * (channels + 1) + 8 * channels * channels * width
                                                           + 4 * tokens * channels * 32)}
    ranks = _ranks(case)
    # The projection and the residual reconstruction; P, codes and rows once.
    return {"bytes": sum(source + 5 * tokens * rank + 2 * rank * channels for rank in ranks),
            "flops": sum(4 * tokens * channels * rank for rank in ranks)}


def tolerance(case):
    if case["kind"] == "restore":
        # The output's rounding, and the product's: fp16 and bf16 products round the coefficients.
        rounding = {"bf16": 2.0 ** -9, "fp16": 2.0 ** -12, "fp32": 2.0 ** -24}[case["out"]]
        product = {"fp16": 2.0 ** -12, "bf16": 2.0 ** -9}.get(case["precision"], 2.0 ** -22)
        if case["source"] == "dense":
            product = 0.0
        return {"rel": 4 * (rounding + product), "max": 16 * (rounding + product)}
    if case["kind"] == "gram":
        return {"rel": 2e-6, "max": 2e-5}
    if case["kind"] == "plan":
        # Directions of an iterative solver, stored in fp16: near-equal singular values mix.
        return {"rel": 2e-2, "max": 0.5, "differ": 0.01}
    # FP64 sums rounded once to fp32; codes move only where a coefficient sits on a code boundary.
    return {"rel": 1e-6, "max": 1e-5, "differ": 1e-4}


# ---------------------------------------------------------------------------------------------
# The same outputs in 64 bits
# ---------------------------------------------------------------------------------------------


def _exact_rope(case, table, values, chunk):
    """``values [N, H, D]`` rotated in interleaved pairs at the chunk's positions, in FP64."""
    cos, sin = table.cos.double().to(DEVICE), table.sin.double().to(DEVICE)
    tokens = _tokens(case)
    rows = _rope_rows(case, chunk)
    if case["rope"] == "dense":
        index = (torch.arange(tokens, device=DEVICE) + rows)[:, None].expand(tokens, cos.shape[1])
    else:
        t = torch.arange(tokens, device=DEVICE)
        plane = case["height"] * case["width"]
        axes = (t // plane + rows[0], t // case["width"] % case["height"] + rows[1], t % case["width"] + rows[2])
        index = torch.cat([axis[:, None].expand(tokens, pairs) for axis, pairs in zip(axes, table.sections)], dim=1)
    c, s = cos.gather(0, index)[:, None], sin.gather(0, index)[:, None]
    even, odd = values[..., 0::2], values[..., 1::2]
    return torch.stack((even * c - odd * s, even * s + odd * c), dim=-1).flatten(-2)


def _exact_restore(case, seed):
    tokens, heads, dim = _tokens(case), case["heads"], case["head_dim"]
    table = _table(case, tokens)
    outputs = []
    for targets in _restore_layers(case, seed):
        for target, (basis, chunks) in enumerate(targets):
            parts = []
            for chunk, (rank, values, scale, offset) in enumerate(chunks):
                x = values.double()
                if scale is not None:
                    x = x * torch.from_numpy(scale).double().to(DEVICE) + torch.from_numpy(offset).double().to(DEVICE)
                if basis is not None:
                    x = x @ basis[:rank].double()
                x = x.view(tokens, heads, dim)
                parts.append(x if target or table is None else _exact_rope(case, table, x, chunk))
            cache = torch.cat(parts)
            outputs.append({"BTHD": cache[None], "THD": cache, "BHTD": cache.transpose(0, 1)[None]}[case["layout"]])
    return outputs


def exact(case, seed):
    if case["kind"] == "restore":
        return _exact_restore(case, seed)
    if case["kind"] == "plan":
        return None  # an iterative solver's directions at a rank it decides itself
    matrices = _sources(case, seed)
    if case["kind"] == "gram":
        return torch.stack([x.double().T @ x.double() for x in matrices])
    if case["kind"] == "tile":
        x = matrices[0].double()
        basis = _orthonormal(case["rank"], case["channels"], _generator(seed, 2), torch.float16).double()
        p = x @ basis.T
        residual = x - p.float().double() @ basis
        return {"coefficients": p, "codes": None, "affine": None, "residual": float(residual.norm() / x.norm()),
                "norm": float(x.norm())}
    stored, span, source = [], [], []
    for matrix, rows in zip(matrices, _bases(case, matrices, seed)):
        x, q = matrix.double(), rows.double()
        p = (x @ q.T).float().double()
        energy = float(x.square().sum())
        stored.append(1.0 - float((x - p @ q).square().sum()) / energy)
        span.append(float((torch.linalg.solve(q @ q.T, p.T @ p)).diagonal().sum()) / energy)
        source.append(energy)
    return {"codes": None, "affine": None, "stored": np.array(stored), "span": np.array(span), "source": np.array(source)}
