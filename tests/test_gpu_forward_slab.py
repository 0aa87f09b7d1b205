"""The forward that keeps a slab's coarse levels in LDS (msda_forward_slab), on
shapes large enough to take it, against the row kernel and the oracle.

Every query is independent, so the same call cut into runs of 200 queries --
too few for the slab kernel -- gives the row kernel's result for all of them. In
float32 both are within 1e-5 (the forward's parity bar: 128 products of unit
weights and values around 1, 128 * 2^-24 * 1 = 8e-6 at worst); 16-bit results
differ by at most one rounding step where the float32 sums round apart.
"""

from __future__ import annotations

import pytest
import torch

from conftest import gpu_available
from muspace_amd import multi_scale_deformable_attn
from muspace_amd.ops.msda_softmax import multi_scale_deformable_attn_softmax
from muspace_amd.ops.scatter_div import multi_scale_deformable_attn_scatter_div
from muspace_amd.runtime.native import load_native_module
from oracle import msda_torch

pytestmark = [
    pytest.mark.gpu,
    pytest.mark.skipif(not gpu_available(), reason="AMD GPU required"),
]

DEV = "cuda"
PIECE = 200
STEP = {torch.float32: 0.0, torch.float16: 2.0**-10, torch.bfloat16: 2.0**-7}


def _inputs(seed, levels, queries, points, heads=8, channels=32, batch=1, vdt=torch.float32,
            gdt=torch.float32):
    g = torch.Generator().manual_seed(seed)
    nv = sum(h * w for h, w in levels)
    value = torch.randn(batch, nv, heads, channels, generator=g).to(vdt)
    loc = torch.rand(batch, queries, heads, len(levels), points, 2, generator=g) * 1.2 - 0.1
    loc.view(-1)[:: 997] = float("nan")
    logits = torch.randn(batch, queries, heads, len(levels) * points, generator=g)
    starts = [0]
    for h, w in levels[:-1]:
        starts.append(starts[-1] + h * w)
    return (value.to(DEV), torch.tensor(levels, device=DEV),
            torch.tensor(starts, device=DEV), loc.to(gdt).to(DEV),
            logits.view(batch, queries, heads, len(levels), points).to(DEV))


def _weights(logits, gdt):
    return logits.flatten(3).softmax(-1).view_as(logits).to(gdt)


def _by_rows(value, shapes, starts, loc, attn):
    return torch.cat([
        multi_scale_deformable_attn(value, shapes, starts, loc[:, q: q + PIECE].contiguous(),
                                    attn[:, q: q + PIECE].contiguous())
        for q in range(0, loc.shape[1], PIECE)], 1)


def _compare(actual, expected):
    tol = STEP[actual.dtype]
    torch.testing.assert_close(actual.float(), expected.float(), rtol=tol, atol=1e-5 + tol * 0.05)


F32, F16, BF16 = torch.float32, torch.float16, torch.bfloat16
CASES = [
    # (levels, queries, points, heads, channels, batch, value, geometry): what is kept in LDS
    (((30, 40), (15, 20), (8, 10), (4, 5)), 5921, 8, 8, 32, 1, F32, F32),  # the last three levels
    (((12, 16), (6, 8), (3, 4), (2, 2)), 8200, 4, 8, 32, 1, F32, F32),     # every level
    (((90, 100), (70, 80)), 8201, 8, 8, 32, 1, F32, F32),                  # none
    (((4, 5), (8, 10), (60, 70)), 5500, 8, 8, 32, 1, F32, F32),            # none: fine level last
    (((60, 70), (30, 35), (1, 1), (1, 2)), 6600, 5, 8, 32, 1, F32, F32),   # 20 samples
    (((60, 70), (30, 35), (15, 18)), 15000, 3, 8, 32, 1, F32, F32),        # 9 samples: ragged stages
    (((60, 70), (30, 35)), 32768, 2, 8, 32, 1, F32, F32),                  # 4 samples, whole rounds
    (((60, 70), (30, 35)), 33000, 2, 8, 32, 1, F16, F32),                  # 4 samples
    (((40, 50), (20, 25), (10, 13), (5, 7)), 7650, 8, 8, 32, 1, BF16, F32),
    (((40, 50), (20, 25), (10, 13), (5, 7)), 7999, 8, 8, 32, 1, F16, F16),
    (((60, 70), (30, 35), (15, 18)), 7500, 4, 8, 32, 3, F16, F32),         # 12 samples
    (((60, 70), (30, 35), (15, 18)), 15000, 3, 8, 32, 1, BF16, BF16),      # 9 samples, 16-bit pairs
    (((40, 50), (20, 25), (10, 13), (5, 7)), 8300, 8, 4, 64, 1, F32, F32),
    (((40, 50), (20, 25), (10, 13)), 22000, 4, 4, 64, 1, BF16, F32),
    (((70, 80),), 70001, 4, 8, 32, 1, F32, F32),                           # one level
    (((70, 80),), 70001, 5, 8, 32, 1, F16, F32),
    (((70, 80),), 35000, 8, 4, 64, 2, BF16, BF16),
]


@pytest.mark.parametrize("case", CASES, ids=[
    f"{len(c[0])}x{c[2]}-q{c[1]}-m{c[3]}c{c[4]}b{c[5]}-{str(c[6])[6:]}-{str(c[7])[6:]}" for c in CASES])
def test_matches_the_row_kernel_and_the_oracle(case):
    levels, queries, points, heads, channels, batch, vdt, gdt = case
    value, shapes, starts, loc, logits = _inputs(5, levels, queries, points, heads, channels,
                                                 batch, vdt, gdt)
    attn = _weights(logits, gdt)
    lib = load_native_module()
    assert lib.forward_takes_slab(value, loc) and not lib.forward_takes_slab(value, loc[:, :PIECE])
    out = multi_scale_deformable_attn(value, shapes, starts, loc, attn)
    _compare(out, _by_rows(value, shapes, starts, loc, attn))
    pick = torch.arange(0, queries, queries // 40)
    some = loc[:, pick].cpu().float()
    some = torch.where(torch.isnan(some).any(-1, keepdim=True), torch.full_like(some, -9.0), some)
    ref = msda_torch.msda_forward(value.cpu().float(), shapes.cpu(), some,
                                  attn[:, pick].cpu().float())
    tol = 1e-5 if vdt == F32 else 1e-2
    torch.testing.assert_close(out[:, pick].cpu().float(), ref, rtol=tol, atol=tol)


@pytest.mark.parametrize("vdt", [F32, F16])
def test_bad_levels_contribute_nothing(vdt):
    """A level past the value and one that overlaps another, among the LDS levels."""
    value, shapes, starts, loc, logits = _inputs(6, ((30, 40), (15, 20), (8, 10), (4, 5)), 7900, 8,
                                                 vdt=vdt)
    assert load_native_module().forward_takes_slab(value, loc)
    starts = starts.clone()
    starts[2] = 1200  # inside level 1
    starts[3] = value.shape[1] - 3
    attn = _weights(logits, F32)
    _compare(multi_scale_deformable_attn(value, shapes, starts, loc, attn),
             _by_rows(value, shapes, starts, loc, attn))


@pytest.mark.parametrize("vdt", [F32, BF16])
@pytest.mark.parametrize("lens", [(7900, 7900, 7600), (7900, 0, 17)])
@pytest.mark.parametrize("levels", [((30, 40), (15, 20), (8, 10), (4, 5)), ((30, 40),)],
                         ids=["four", "one"])
def test_camera_average(vdt, lens, levels):
    """Cameras of unequal length (one empty) into BEV slots, an index out of range.
    With one level cameras keep the row kernel."""
    cams, nq = len(lens), 9000
    value, shapes, starts, loc, logits = _inputs(7, levels, 7900, 8, batch=cams, vdt=vdt)
    assert (load_native_module().forward_takes_slab(value[:1], loc[:1, : max(lens)], cams)
            == (len(levels) > 1))
    attn = _weights(logits, F32)
    g = torch.Generator().manual_seed(8)
    indexes = [torch.randperm(nq, generator=g)[:n].to(DEV) for n in lens]
    indexes[0][5] = nq + 3
    count = torch.randint(1, 4, (1, nq), generator=g).float().to(DEV)
    with torch.no_grad():
        slots = multi_scale_deformable_attn_scatter_div(value, shapes, starts, loc, attn, indexes,
                                                        count)
        rows = _by_rows(value.float(), shapes, starts, loc, attn)
    ref = torch.zeros(1, nq, 256, device=DEV)
    for cam, index in enumerate(indexes):
        ok = index < nq
        ref[0, index[ok]] += rows[cam, : len(index)][ok] / count[0, index[ok]].unsqueeze(-1)
    tol = 1e-5 if vdt == F32 else 2e-2
    torch.testing.assert_close(slots.float(), ref, rtol=tol, atol=tol)


@pytest.mark.parametrize("vdt,gdt", [(F32, F32), (BF16, F32), (F16, F16)])
@pytest.mark.parametrize("softmax", [False, True])
def test_training_calls_that_bin_apart(vdt, gdt, softmax):
    """Output and gradients of a call whose forward takes the slab kernel after the
    binning kernels, against runs of few queries (grad_value: their sum)."""
    levels, queries = ((40, 50), (20, 25), (10, 13)), 11000
    value, shapes, starts, loc, logits = _inputs(9, levels, queries, 4, vdt=vdt, gdt=gdt)
    op = multi_scale_deformable_attn_softmax if softmax else multi_scale_deformable_attn
    weights = logits.to(gdt) if softmax else _weights(logits, gdt)
    grad = torch.randn(1, queries, 256, generator=torch.Generator().manual_seed(10)).to(vdt).to(DEV)

    def call(q0, q1):
        leaves = [t.clone().requires_grad_() for t in
                  (value, loc[:, q0:q1], weights[:, q0:q1])]
        out = op(leaves[0], shapes, starts, leaves[1], leaves[2])
        return (out.detach(), *torch.autograd.grad(out, leaves, grad[:, q0:q1]))

    whole = call(0, queries)
    pieces = [call(q, min(q + 500, queries)) for q in range(0, queries, 500)]
    _compare(whole[0], torch.cat([p[0] for p in pieces], 1))
    gv = sum(p[1].float() for p in pieces)
    tol = 1e-4 if vdt == F32 else 2e-2
    torch.testing.assert_close(whole[1].float(), gv, rtol=tol, atol=tol * gv.abs().max().item())
    for i in (2, 3):
        piece = torch.cat([p[i] for p in pieces], 1)
        torch.testing.assert_close(whole[i].float(), piece.float(), rtol=tol, atol=tol)


def test_records_past_the_memory_side_cache():
    """A batch whose binned records pass 256 MB (their stores then go through the L2)
    gives what its entries give one by one. Outputs and location and weight
    gradients are each one unit's or sample's own sum. A value gradient sums, in
    another order, up to some 350 products (20200 queries x 4 samples x 4 corners over
    952 cells) whose magnitudes add up to about 9: 350 * 2^-24 * 9 = 1.9e-4 at worst."""
    levels, queries, points, batch = ((56, 68), (28, 34)), 20200, 4, 13
    value, shapes, starts, loc, logits = _inputs(11, levels, queries, points, batch=batch)
    assert batch * queries * 8 * len(levels) * points * 16 > 256 << 20
    attn = _weights(logits, F32)
    grad = torch.randn(batch, queries, 256, generator=torch.Generator().manual_seed(12)).to(DEV)

    def call(part):
        leaves = [t[part].clone().requires_grad_() for t in (value, loc, attn)]
        out = multi_scale_deformable_attn(leaves[0], shapes, starts, leaves[1], leaves[2])
        return (out.detach(), *torch.autograd.grad(out, leaves, grad[part]))

    whole = call(slice(None))
    for entry in (0, 5, batch - 1):
        one = call(slice(entry, entry + 1))
        for i, atol in enumerate((1e-5, 2e-4, 1e-5, 1e-5)):
            torch.testing.assert_close(whole[i][entry: entry + 1], one[i], rtol=1e-5, atol=atol)
