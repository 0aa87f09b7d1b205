"""Performance cases of the framework: what a user's program has it do, call by call.

Every case goes through a public operator of ``muspace_amd`` (inference: the
call alone; training: the call and its backward through autograd) on inputs
drawn on the GPU from a seed:

  msda          ``multi_scale_deformable_attn``
  msda_softmax  ``multi_scale_deformable_attn_softmax`` (attention logits)
  sca_average   ``multi_scale_deformable_attn_scatter_div`` (cameras -> BEV slots)
  aggregation   ``deformable_aggregation``

Sampling locations follow their use: ``uniform`` (the benchmark configurations'
own draw), ``cells`` (encoder self-attention: query i sits on value cell i),
``grid`` (a BEV grid in row-major order), ``objects`` (decoder queries at
arbitrary places) -- the last three with offsets of a few pixels of the level
they sample -- and, for sca_average, BEV cells projected into a camera ring.
All locations are multiples of 2^-15. A level is at most 256 wide and high, so
location * size - 0.5 is exact in float32 and float64 alike and every correct
implementation sees the same cells: the location gradient jumps from cell to
cell, and would otherwise differ by whole samples where a coordinate rounds onto
a border.
"""

from __future__ import annotations

import math

import torch

from muspace_amd.ops.deformable_aggregation import deformable_aggregation
from muspace_amd.ops.msda_softmax import multi_scale_deformable_attn_softmax
from muspace_amd.ops.multi_scale_deformable_attn import multi_scale_deformable_attn
from muspace_amd.ops.scatter_div import multi_scale_deformable_attn_scatter_div

DEVICE = "cuda"
DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
LOCATION_STEPS = 2.0**15
OFFSET_PIXELS = 3.0  # learned offsets: a few pixels of the sampled level
CAMERA_FOV_DEG = 90.0

DETR_LEVELS = "100x167,50x84,25x42,13x21"
SCA_LEVELS = "116x200,58x100,29x50,15x25"
DRIVE_SCALES = "64x176,32x88,16x44,8x22"


def _msda(name, op, mode, dtype, batch, queries, levels, points, locations, heads=8, channels=32):
    return {
        "name": name, "op": op, "mode": mode, "dtype": dtype, "batch": batch, "queries": queries,
        "heads": heads, "channels": channels, "levels": levels, "points": points,
        "locations": locations,
    }


def listed():
    return [
        # a small model's encoder layer, one image, four tiny levels: the
        # latency of a call
        _msda("small_encoder_infer_f32", "msda", "infer", "float32", 1, 1000,
              "32x32,16x16,8x8,4x4", 4, "uniform"),
        # object decoder cross-attention at serving time: few queries on the
        # maps of one full-size image, half precision
        _msda("decoder_infer_f16", "msda", "infer", "float16", 1, 300, DETR_LEVELS, 4, "objects"),
        # the same layer in training: little sampled, but the whole value's
        # gradient is written
        _msda("decoder_train_f32", "msda", "train", "float32", 2, 900, DETR_LEVELS, 4, "objects"),
        # Deformable-DETR encoder self-attention in training, every cell a query
        _msda("encoder_train_f32", "msda", "train", "float32", 2, 22223, DETR_LEVELS, 4, "cells"),
        # an encoder of another image size and three levels, trained in half
        # precision from attention logits; odd sizes throughout
        _msda("odd_encoder_softmax_train_f16", "msda_softmax", "train", "float16", 3, 10007,
              "75x101,38x51,19x26", 4, "cells"),
        # BEVFormer temporal self-attention in training: one level, a BEV grid
        _msda("tsa_train_f32", "msda", "train", "float32", 2, 40000, "200x200", 4, "grid"),
        # BEVFormer spatial cross-attention: inference in bfloat16 ...
        _msda("sca_infer_bf16", "msda", "infer", "bfloat16", 6, 10000, SCA_LEVELS, 8, "uniform"),
        # ... training in float32 (the benchmark's default workload) ...
        _msda("sca_train_f32", "msda", "train", "float32", 6, 10000, SCA_LEVELS, 8, "uniform"),
        # ... and the largest: two samples, bfloat16 value, float32 geometry
        _msda("sca_train_bf16", "msda", "train", "bfloat16", 12, 15000, SCA_LEVELS, 8, "uniform"),
        # the same attention with the camera average fused, one sample, training
        {"name": "sca_average_train_f32", "op": "sca_average", "mode": "train",
         "dtype": "float32", "batch": 1, "cameras": 6, "bev": 200, "heads": 8, "channels": 32,
         "levels": SCA_LEVELS, "points": 8},
        # SparseDrive's aggregation: one sample when driving ...
        {"name": "aggregation_infer_f32", "op": "aggregation", "mode": "infer",
         "dtype": "float32", "batch": 1, "cameras": 6, "anchors": 900, "points": 13, "groups": 8,
         "channels": 256, "levels": DRIVE_SCALES},
        # ... and a training batch
        {"name": "aggregation_train_f32", "op": "aggregation", "mode": "train",
         "dtype": "float32", "batch": 8, "cameras": 6, "anchors": 900, "points": 13, "groups": 8,
         "channels": 256, "levels": DRIVE_SCALES},
    ]


# Bounds of a drawn case: half the samples of the largest listed one (a sample
# of narrow channels costs no less than one of 32, and float32 up to twice a
# 16-bit one), and its value elements.
MAX_SAMPLE_CHANNELS = 12 * 15000 * 8 * 32 * 32 // 2
MAX_VALUE = 12 * 30825 * 256


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _draw_levels(rng, count, high_h, high_w):
    h, w = _log_uniform(rng, 20, high_h), _log_uniform(rng, 20, high_w)
    sizes = []
    for _ in range(count):
        sizes.append(f"{max(h, 1)}x{max(w, 1)}")
        h, w = (h + 1) // 2, (w + 1) // 2
    return ",".join(sizes)


def draw(rng):
    op = rng.choice(["msda", "msda", "msda", "msda_softmax", "sca_average", "aggregation"])
    mode = rng.choice(["infer", "train"])
    while True:
        if op == "aggregation":
            case = {"op": op, "mode": mode, "dtype": "float32", "batch": rng.randint(1, 8),
                    "cameras": rng.randint(1, 6), "anchors": _log_uniform(rng, 50, 900),
                    "points": rng.randint(5, 13), "groups": 8,
                    "channels": rng.choice([128, 256, 256]),
                    "levels": _draw_levels(rng, rng.randint(2, 4), 64, 176)}
            return case
        dtype = rng.choice(["float32", "float16", "bfloat16"])
        heads, channels = rng.choice([(8, 32), (8, 32), (8, 32), (8, 16), (4, 64), (6, 32)])
        count = rng.randint(1, 5)
        points = rng.choice([2, 3, 4, 4, 5, 8])
        levels = _draw_levels(rng, count, 200, 200)
        if op == "sca_average":
            case = {"op": op, "mode": mode, "dtype": dtype, "batch": 1,
                    "cameras": rng.randint(4, 6), "bev": _log_uniform(rng, 30, 200),
                    "heads": heads, "channels": channels, "levels": levels, "points": points}
        else:
            locations = rng.choice(["uniform", "cells", "grid", "objects"])
            queries = _log_uniform(rng, 100, 40000)
            if locations == "cells":
                queries = sum(h * w for h, w in _sizes({"levels": levels}))
            if locations == "objects":
                queries = min(queries, 1500)
            case = {"op": op, "mode": mode, "dtype": dtype, "batch": _log_uniform(rng, 1, 12),
                    "queries": queries, "heads": heads, "channels": channels, "levels": levels,
                    "points": points, "locations": locations}
        rows, spatial = _rows_and_spatial(case)
        samples = rows * heads * count * points
        value = _slabs(case) * spatial * heads * channels
        if samples * max(channels, 32) <= MAX_SAMPLE_CHANNELS and value <= MAX_VALUE:
            return case


# -------------------------------------------------------------- sizes ---


def _sizes(case):
    return [tuple(int(n) for n in level.split("x")) for level in case["levels"].split(",")]


def _slabs(case):
    return case["batch"] * case.get("cameras", 1)


def _camera_cells(case):
    """Per camera of a ring around a bev x bev grid: the cells it sees, their
    angle from its axis in degrees and their distance from the centre."""
    n = case["bev"]
    axis = torch.arange(n, dtype=torch.float64) + 0.5 - n / 2
    ys, xs = torch.meshgrid(axis, axis, indexing="ij")
    angle = torch.rad2deg(torch.atan2(ys, xs)).flatten()
    distance = torch.sqrt(xs * xs + ys * ys).flatten()
    cameras = []
    for cam in range(case["cameras"]):
        off = (angle - 360.0 * cam / case["cameras"] + 180.0) % 360.0 - 180.0
        seen = torch.nonzero(off.abs() < CAMERA_FOV_DEG / 2).flatten()
        cameras.append((seen, off[seen], distance[seen]))
    return cameras


def _rows_and_spatial(case):
    """(query rows over the batch, value cells of one slab)."""
    spatial = sum(h * w for h, w in _sizes(case))
    if case["op"] == "sca_average":
        return case["batch"] * sum(len(seen) for seen, _, _ in _camera_cells(case)), spatial
    return case["batch"] * case["queries"], spatial


def work(case):
    sizes = _sizes(case)
    spatial = sum(h * w for h, w in sizes)
    train = case["mode"] == "train"
    width = 4 if case["dtype"] == "float32" else 2
    if case["op"] == "aggregation":
        batch, channels = case["batch"], case["channels"]
        feat = batch * case["cameras"] * spatial * channels
        pairs = batch * case["anchors"] * case["points"] * case["cameras"]
        weights = pairs * len(sizes) * case["groups"]
        out = batch * case["anchors"] * channels
        moved = feat + 2 * pairs + weights + out
        if train:
            moved += out + feat + 2 * pairs + weights
        flops = pairs * ACTIVE_SHARE * len(sizes) * 4 * channels * 2
        return {"bytes": 4 * moved, "flops": int(flops * (3 if train else 1))}
    rows, spatial = _rows_and_spatial(case)
    heads, channels = case["heads"], case["channels"]
    value = _slabs(case) * spatial * heads * channels
    samples = rows * heads * len(sizes) * case["points"]
    out = rows * heads * channels
    extra = 0
    if case["op"] == "sca_average":
        out = case["batch"] * case["bev"] ** 2 * heads * channels
        extra = 8 * (rows // case["batch"]) + 4 * case["batch"] * case["bev"] ** 2
    moved = width * (value + out) + 4 * 3 * samples + extra
    if train:  # grad_output in; the gradients out, each in its input's type
        moved += width * (out + value) + 4 * 3 * samples
    flops = samples * 4 * channels * 2
    return {"bytes": moved, "flops": flops * (3 if train else 1)}


# ------------------------------------------------------------- inputs ---


def _snap(loc):
    return torch.round(loc * LOCATION_STEPS) / LOCATION_STEPS


def _level_scale(sizes):
    """(W, H) per level, broadcast over [.., L, P, 2]."""
    return torch.tensor([[w, h] for h, w in sizes], dtype=torch.float32,
                        device=DEVICE).view(len(sizes), 1, 2)


def _references(case, sizes, gen):
    """Reference points [batch or 1, queries, 2] in [0, 1]."""
    queries = case["queries"]
    if case["locations"] == "objects":
        return torch.rand((case["batch"], queries, 2), generator=gen, device=DEVICE)
    if case["locations"] == "cells":
        grids = sizes
    else:
        cols = math.isqrt(queries - 1) + 1
        grids = [((queries + cols - 1) // cols, cols)]
    points = []
    for h, w in grids:
        ys, xs = torch.meshgrid((torch.arange(h, device=DEVICE) + 0.5) / h,
                                (torch.arange(w, device=DEVICE) + 0.5) / w, indexing="ij")
        points.append(torch.stack([xs, ys], -1).view(-1, 2))
    return torch.cat(points)[:queries].unsqueeze(0)


def _geometry(case, seed):
    """Everything but value and grad_output, in float32, from the seed."""
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    sizes = _sizes(case)
    heads, levels, points = case["heads"], len(sizes), case["points"]
    if case["op"] == "sca_average":
        cameras = _camera_cells(case)
        rows = max(len(seen) for seen, _, _ in cameras)
        slabs = _slabs(case)
        # azimuth across the image, four pillar heights down it
        ref = torch.full((case["cameras"], rows, points, 2), 0.5, dtype=torch.float64)
        heights = torch.arange(points, dtype=torch.float64) % 4 - 1.0
        for cam, (seen, off, distance) in enumerate(cameras):
            ref[cam, : len(seen), :, 0] = (0.5 + off / CAMERA_FOV_DEG).view(-1, 1)
            ref[cam, : len(seen), :, 1] = (
                0.5 + heights.view(1, -1) * case["bev"] / 20 / (distance.view(-1, 1) + 5.0))
        centre = ref.float().to(DEVICE).view(1, case["cameras"], rows, 1, 1, points, 2)
        shape = (case["batch"], case["cameras"], rows, heads, levels, points, 2)
        offset = torch.randn(shape, generator=gen, device=DEVICE) * OFFSET_PIXELS
        loc = (centre + offset / _level_scale(sizes)).view(slabs, rows, heads, levels, points, 2)
        queries = rows
    else:
        slabs, queries = case["batch"], case["queries"]
        shape = (slabs, queries, heads, levels, points, 2)
        if case["locations"] == "uniform":
            loc = torch.rand(shape, generator=gen, device=DEVICE) * 1.035 - 0.0175
        else:
            centre = _references(case, sizes, gen).view(-1, queries, 1, 1, 1, 2)
            offset = torch.randn(shape, generator=gen, device=DEVICE) * OFFSET_PIXELS
            loc = centre + offset / _level_scale(sizes)
    loc = _snap(loc.clamp_(-0.05, 1.05))
    logits = torch.randn((slabs, queries, heads, levels * points), generator=gen, device=DEVICE)
    weights = logits if case["op"] == "msda_softmax" else logits.softmax(-1)
    return gen, loc, weights.view(slabs, queries, heads, levels, points)


ACTIVE_SHARE = 0.186  # (anchor, point, camera) triples that fall inside an image


def _aggregation_inputs(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    sizes = _sizes(case)
    spatial, cams = sum(h * w for h, w in sizes), case["cameras"]
    triples = (case["batch"], case["anchors"], case["points"], cams)
    feat = torch.randn((case["batch"], cams * spatial, case["channels"]), generator=gen,
                       device=DEVICE)
    active = torch.rand(triples, generator=gen, device=DEVICE) < ACTIVE_SHARE
    outside = torch.randn((*triples, 2), generator=gen, device=DEVICE) * 10.0
    inside = torch.rand((*triples, 2), generator=gen, device=DEVICE) * 0.98 + 0.01
    loc = _snap(torch.where(active.unsqueeze(-1), inside, outside))
    weights = torch.rand((*triples, len(sizes), case["groups"]), generator=gen,
                         device=DEVICE) * 0.004
    starts, at = [], 0
    for _ in range(cams):
        row = []
        for h, w in sizes:
            row.append(at)
            at += h * w
        starts.append(row)
    grad = torch.randn((case["batch"], case["anchors"], case["channels"]), generator=gen,
                       device=DEVICE)
    return {
        "feat": feat,
        "shapes": torch.tensor([[list(s) for s in sizes]] * cams, dtype=torch.int32,
                               device=DEVICE),
        "starts": torch.tensor(starts, dtype=torch.int32, device=DEVICE),
        "loc": loc, "weights": weights, "grad": grad,
    }


def _inputs(case, seed):
    """A case's tensors, before any requires a gradient."""
    if case["op"] == "aggregation":
        return _aggregation_inputs(case, seed)
    dtype = DTYPES[case["dtype"]]
    sizes = _sizes(case)
    heads, channels = case["heads"], case["channels"]
    gen, loc, weights = _geometry(case, seed)
    slabs, queries = loc.shape[:2]
    cells = [h * w for h, w in sizes]
    starts = [sum(cells[:i]) for i in range(len(cells))]
    value = torch.randn((slabs, sum(cells), heads, channels), generator=gen, device=DEVICE)
    state = {
        "value": value.to(dtype),
        "shapes": torch.tensor(sizes, dtype=torch.int64, device=DEVICE),
        "starts": torch.tensor(starts, dtype=torch.int64, device=DEVICE),
        "loc": loc, "weights": weights,
    }
    rows = (slabs, queries)
    if case["op"] == "sca_average":
        cameras = _camera_cells(case)
        bev = case["bev"] ** 2
        count = torch.zeros(bev)
        for seen, _, _ in cameras:
            count[seen] += 1
        state["indexes"] = [seen.to(DEVICE) for seen, _, _ in cameras]
        state["count"] = count.clamp(min=1).repeat(case["batch"], 1).to(DEVICE)
        rows = (case["batch"], bev)
    state["grad"] = torch.randn((*rows, heads * channels), generator=gen,
                                device=DEVICE).to(dtype)
    return state


def prepare(case, seed):
    state = _inputs(case, seed)
    state["op"], state["train"] = case["op"], case["mode"] == "train"
    if state["train"]:
        for name in ("feat", "value", "loc", "weights"):
            if name in state:
                state[name].requires_grad_()
    return state


def _call(state):
    op = state["op"]
    if op == "aggregation":
        return deformable_aggregation(state["feat"], state["shapes"], state["starts"],
                                      state["loc"], state["weights"])
    args = (state["value"], state["shapes"], state["starts"], state["loc"], state["weights"])
    if op == "msda":
        return multi_scale_deformable_attn(*args)
    if op == "msda_softmax":
        return multi_scale_deformable_attn_softmax(*args)
    return multi_scale_deformable_attn_scatter_div(*args, state["indexes"], state["count"])


def run(state):
    if not state["train"]:
        with torch.no_grad():
            return _call(state)
    out = _call(state)
    source = state["feat"] if state["op"] == "aggregation" else state["value"]
    grads = torch.autograd.grad(out, (source, state["loc"], state["weights"]), state["grad"])
    return (out.detach(), *grads)


# ---------------------------------------------------------- tolerance ---


def tolerance(case):
    # relative 2-norm errors against 64 bits measure 4e-8 to 1.3e-7 in float32
    # (the order of the sums) and, in 16 bits, the rounding of the results
    # themselves: 1.7e-3 in bfloat16, 2.1e-4 in float16. Four times these (float32:
    # eight, for sums split in other ways over longer inputs)
    if case["dtype"] == "float32":
        return {"rel": 1e-6}
    if case["dtype"] == "bfloat16":
        return {"rel": 7e-3}
    return {"rel": 9e-4}


# ------------------------------------------------------------- 64 bits ---


def _corners(loc, h, w):
    """The four bilinear corners of float64 locations [..., 2] on an h x w map:
    (cell, inside, weight, d weight / d x, d weight / d y), x and y in [0, 1]."""
    x, y = loc[..., 0] * w - 0.5, loc[..., 1] * h - 0.5
    x0, y0 = torch.floor(x), torch.floor(y)
    fx, fy = x - x0, y - y0
    for dy in (0, 1):
        for dx in (0, 1):
            cx, cy = x0 + dx, y0 + dy
            inside = (cx >= 0) & (cx < w) & (cy >= 0) & (cy < h)
            cell = cy.clamp(0, h - 1).long() * w + cx.clamp(0, w - 1).long()
            wx, wy = (fx if dx else 1 - fx), (fy if dy else 1 - fy)
            keep = inside.double()
            yield (cell, inside, wx * wy * keep, (w if dx else -w) * wy * keep,
                   (h if dy else -h) * wx * keep)


def _exact_slab(value, loc, weights, sizes, grad):
    """One (batch entry, head) in float64: value [nv, C], loc [n, L, P, 2],
    weights [n, L, P], grad [n, C] or None. Returns (out, grads or None)."""
    out = value.new_zeros((loc.shape[0], value.shape[1]))
    grad_value = torch.zeros_like(value)
    grad_loc, grad_weights = torch.zeros_like(loc), torch.zeros_like(weights)
    start = 0
    for level, (h, w) in enumerate(sizes):
        a = weights[:, level]
        for cell, inside, wgt, dx, dy in _corners(loc[:, level], h, w):
            rows = value[start + cell]  # [n, P, C]
            coef = a * wgt
            out += (coef.unsqueeze(-1) * rows).sum(1)
            if grad is not None:
                dot = (rows * grad.unsqueeze(1)).sum(-1)
                grad_weights[:, level] += wgt * dot
                grad_loc[:, level, :, 0] += a * dx * dot
                grad_loc[:, level, :, 1] += a * dy * dot
                add = (coef.unsqueeze(-1) * grad.unsqueeze(1)).flatten(0, 1)
                grad_value.index_put_((start + cell.flatten(),), add, accumulate=True)
        start += h * w
    return out, (grad_value, grad_loc, grad_weights) if grad is not None else None


def _exact_msda(case, state):
    sizes = _sizes(case)
    value, loc, weights = (state[k].double() for k in ("value", "loc", "weights"))
    train = case["mode"] == "train"
    slabs, queries, heads = weights.shape[:3]
    channels = value.shape[3]
    softmax = case["op"] == "msda_softmax"
    if softmax:
        weights = weights.flatten(3).softmax(-1).view_as(weights)
    average = case["op"] == "sca_average"
    if average:
        slots = state["grad"].new_zeros(state["grad"].shape, dtype=torch.float64)
        scale = (1.0 / state["count"].double()).unsqueeze(-1)
        grad_slots = state["grad"].double() * scale
    out = value.new_zeros((slabs, queries, heads * channels))
    grads = tuple(torch.zeros_like(t) for t in (value, loc, weights))
    for b in range(slabs):
        n, seen, entry = queries, None, b
        if average:
            entry, cam = divmod(b, case["cameras"])
            seen = state["indexes"][cam]
            n = len(seen)
        for m in range(heads):
            part = slice(m * channels, (m + 1) * channels)
            grad = None
            if train:
                grad = grad_slots[entry, seen, part] if average \
                    else state["grad"][b, :, part].double()
            row, slab = _exact_slab(value[b, :, m], loc[b, :n, m], weights[b, :n, m], sizes, grad)
            out[b, :n, part] = row
            if train:
                grads[0][b, :, m] = slab[0]
                grads[1][b, :n, m] = slab[1]
                grads[2][b, :n, m] = slab[2]
        if average:
            slots[entry, seen] += out[b, :n] * scale[entry, seen]
    if softmax and train:
        mean = (grads[2] * weights).flatten(3).sum(-1)[..., None, None]
        grads = (grads[0], grads[1], weights * (grads[2] - mean))
    out = slots if average else out
    return (out, *grads) if train else out


def _exact_aggregation(case, state):
    sizes, train = _sizes(case), case["mode"] == "train"
    feat, loc, weights, grad = (state[k].double() for k in ("feat", "loc", "weights", "grad"))
    channels, groups = case["channels"], case["groups"]
    out = torch.zeros_like(grad)
    grads = tuple(torch.zeros_like(t) for t in (feat, loc, weights))
    x, y = loc[..., 0], loc[..., 1]
    active = (x > 0) & (x < 1) & (y > 0) & (y < 1)
    for b in range(case["batch"]):
        for cam in range(case["cameras"]):
            anchor, point = torch.nonzero(active[b, :, :, cam], as_tuple=True)
            where = loc[b, anchor, point, cam]
            g = grad[b, anchor]
            for scale, (h, w) in enumerate(sizes):
                start = cam * sum(a * c for a, c in sizes)
                start += sum(a * c for a, c in sizes[:scale])
                part = weights[b, anchor, point, cam, scale]  # [n, groups]
                wide = part.repeat_interleave(channels // groups, -1)
                gw = g * wide
                gl, gp = torch.zeros_like(where), torch.zeros_like(part)
                for cell, inside, wgt, dx, dy in _corners(where, h, w):
                    rows = feat[b, start + cell]
                    out[b].index_put_((anchor,), wgt.unsqueeze(-1) * wide * rows, accumulate=True)
                    if train:
                        dot = (rows * g).view(-1, groups, channels // groups).sum(-1)
                        gp += wgt.unsqueeze(-1) * dot
                        along = (dot * part).sum(-1)
                        gl[:, 0] += dx * along
                        gl[:, 1] += dy * along
                        grads[0][b].index_put_((start + cell,), wgt.unsqueeze(-1) * gw,
                                               accumulate=True)
                if train:
                    grads[1][b, anchor, point, cam] += gl
                    grads[2][b, anchor, point, cam, scale] = gp
    return (out, *grads) if train else out


def exact(case, seed):
    state = _inputs(case, seed)
    with torch.no_grad():
        if case["op"] == "aggregation":
            return _exact_aggregation(case, state)
        return _exact_msda(case, state)
