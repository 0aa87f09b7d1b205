"""Feature gradients of deformable aggregation summed by owner (the operator's
backward, deformable_aggregation_backward_ws): where its counting sort and its
split of a row among wavefronts can go wrong, against the float64 oracle.

The sums are float64 over exact products of float32 factors, rounded once; the
factors (a bilinear weight, grad_output times a weight) carry one or two
float32 roundings each, so an element is within 4 * 2^-24 of the sum of its
contributions' magnitudes. Locations sit on a 1/4096 grid, where the float32
cell coordinates are exact.
"""

from __future__ import annotations

import pytest
import torch

from conftest import gpu_available
from muspace_amd.runtime.native import load_native_module
from oracle import dfa_torch
from test_dfa_oracle import random_case



def gpu(test):
    return pytest.mark.gpu(pytest.mark.skipif(not gpu_available(), reason="AMD GPU required")(test))


DEV = "cuda"


def _case(seed, shapes, channels, groups, anchors, batch=2, pts=3, cams=3):
    case = list(random_case(seed, batch=batch, anchors=anchors, pts=pts, cams=cams, shapes=shapes,
                            channels=channels, groups=groups, dtype=torch.float32))
    case[3].copy_(torch.round(case[3] * 4096) / 4096)
    return case


def _dims(case):
    """batch, cams, feat, embeds, scales, anchors, pts, groups"""
    (batch, feat, embeds), weights = case[0].shape, case[4].shape
    return [batch, weights[3], feat, embeds, weights[4], weights[1], weights[2], weights[5]]


def _by_owner(case, grad_out):
    """The sums by owner, with their workspace, also where the operator has the
    atomic kernels for the faster ones."""
    mc, spatial, start, loc, weights = [t.to(DEV) for t in case]
    grad_out = grad_out.to(DEV)
    grads = [torch.full_like(t, float("nan")) for t in (mc, loc, weights)]
    lib, dims = load_native_module(), _dims(case)
    size = lib.raw("deformable_aggregation_backward_workspace_size")(*dims)
    assert size > 0
    workspace = torch.empty(size, dtype=torch.uint8, device=DEV)
    code = lib.raw("deformable_aggregation_backward_ws")(
        *[t.data_ptr() for t in (mc, spatial, start, loc, weights, grad_out, *grads)], *dims,
        workspace.data_ptr(), size, torch.cuda.current_stream().cuda_stream)
    assert code == 0
    return [g.cpu() for g in grads]


def _backward(case, grad_out, name="deformable_aggregation_backward"):
    if name == "deformable_aggregation_backward":
        return _by_owner(case, grad_out)
    mc, spatial, start, loc, weights = [t.to(DEV) for t in case]
    grads = [torch.zeros_like(t) for t in (mc, loc, weights)]
    getattr(load_native_module(), name)(mc, spatial, start, loc, weights, grad_out.to(DEV), *grads)
    return [g.cpu() for g in grads]


def _operator_backward(case, grad_out):
    """As the operator calls it: scratch where the library asks for it."""
    case = [t.to(DEV) for t in case]
    grads = [torch.full_like(case[i], float("nan")) for i in (0, 3, 4)]
    load_native_module().deformable_aggregation_backward(*case, grad_out.to(DEV), *grads)
    return [g.cpu() for g in grads]


def _oracle(case, grad_out):
    ref = [t.double().requires_grad_(True) if t.is_floating_point() else t for t in case]
    (dfa_torch.aggregate_batched(*ref) * grad_out.double()).sum().backward()
    return [ref[i].grad for i in (0, 3, 4)]


def _check(case, grad_out):
    actual, expected = _backward(case, grad_out), _oracle(case, grad_out)
    magnitude = _oracle([case[0], *case[1:4], case[4].abs()], grad_out.abs())[0]
    assert ((actual[0].double() - expected[0]).abs() <= 4 * 2.0**-24 * magnitude + 1e-30).all()
    torch.testing.assert_close(actual[1].double(), expected[1], rtol=1e-4, atol=1e-3)
    torch.testing.assert_close(actual[2].double(), expected[2], rtol=1e-4, atol=1e-4)


# one to four channel slots; feature rows: fewer than a workgroup's 16, not a
# multiple of 16, one range of 2048 and a part of the next, several ranges
@pytest.mark.parametrize("channels,groups", [(64, 8), (128, 4), (192, 3), (256, 8), (256, 1)])
@pytest.mark.parametrize("shapes", [((2, 2),), ((7, 9), (3, 5)), ((25, 28), (2, 2), (1, 1)),
                                    ((64, 44), (32, 22), (16, 11))])
@gpu
def test_row_ranges_and_channel_layouts(channels, groups, shapes):
    case = _case(31, shapes, channels, groups, anchors=40)
    _check(case, torch.randn(2, 40, channels, generator=torch.Generator().manual_seed(32)))


@gpu
@pytest.mark.parametrize("shapes,batch,anchors", [
    (((64, 88), (32, 44)), 2, 40),   # 42240 rows: ranges of 512; 16 rows a workgroup of the sums
    (((100, 90), (50, 45)), 2, 40),  # 67500 rows: ranges of 1024
    (((150, 160), (75, 80)), 2, 40),  # 180000 rows: ranges of 2048
    (((25, 28), (13, 14)), 2, 60),   # 16 rows a workgroup of the sums, 8, 4, 2, 1
    (((25, 28), (13, 14)), 2, 300),
    (((25, 28), (13, 14)), 2, 500),
    (((25, 28), (13, 14)), 2, 900),
    (((25, 28), (13, 14)), 2, 1400),
])
def test_ranges_and_blocks_of_the_sums_by_shape(shapes, batch, anchors):
    case = _case(47, shapes, 128, 8, anchors=anchors, batch=batch, pts=4)
    _check(case, torch.randn(batch, anchors, 128, generator=torch.Generator().manual_seed(48)))


@gpu
@pytest.mark.parametrize("channels,shapes", [(64, ((7, 9), (3, 5))), (256, ((7, 9),))])
def test_operator_with_and_without_scratch(channels, shapes):
    """One scale takes the kernels with atomics."""
    case = _case(49, shapes, channels, 8, anchors=50)
    grad_out = torch.randn(2, 50, channels, generator=torch.Generator().manual_seed(50))
    for g, e, atol in zip(_operator_backward(case, grad_out), _by_owner(case, grad_out),
                          (1e-5, 1e-3, 1e-4)):
        torch.testing.assert_close(g, e, rtol=1e-5, atol=atol)


@gpu
@pytest.mark.parametrize("where", [(0.5, 0.5), (0.02, 0.02), (0.99, 0.5)])
def test_rows_shared_by_wavefronts(where):
    """Every point of every anchor at one place: a few rows take thousands of
    contributions, over all four wavefronts of their workgroup."""
    case = _case(33, ((9, 13), (4, 6), (1, 1)), 256, 8, anchors=333)
    case[3][...] = torch.tensor([round(w * 4096) / 4096 for w in where])
    _check(case, torch.randn(2, 333, 256, generator=torch.Generator().manual_seed(34)))


@gpu
def test_overlapping_and_out_of_range_maps():
    """Maps that share rows list all their contributions there; a map past
    num_feat adds nothing; rows of no map are zero."""
    case = _case(35, ((6, 8), (4, 5)), 128, 8, anchors=50)
    start = case[2]
    start[0, 1] = start[0, 0] + 7  # camera 0: the second map inside the first
    start[1, 0] = case[0].shape[1] - 10  # camera 1: its first map would leave the features
    grad_out = torch.randn(2, 50, 128, generator=torch.Generator().manual_seed(36))
    actual, base = (_backward(case, grad_out, f"deformable_aggregation_backward{suffix}")
                    for suffix in ("", "_base"))
    torch.testing.assert_close(actual[0], base[0], rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(actual[1], base[1], rtol=1e-4, atol=1e-3)
    torch.testing.assert_close(actual[2], base[2], rtol=1e-4, atol=1e-4)


@gpu
def test_non_finite_gradients_and_weights():
    """inf and NaN reach the elements that the base kernels give them."""
    case = _case(37, ((9, 13), (4, 6)), 256, 8, anchors=60)
    case[4][0, 3, 1, 2, 0, 5] = float("inf")
    grad_out = torch.randn(2, 60, 256, generator=torch.Generator().manual_seed(38))
    grad_out[0, 5, 40] = float("inf")
    grad_out[1, 9, 3] = float("nan")
    actual, base = (_backward(case, grad_out, f"deformable_aggregation_backward{suffix}")
                    for suffix in ("", "_base"))
    assert not torch.isfinite(base[0]).all()
    for a, b, atol in zip(actual, base, (1e-4, 1e-3, 1e-4)):
        torch.testing.assert_close(a, b, rtol=1e-4, atol=atol, equal_nan=True)


@gpu
def test_no_active_point():
    """Nothing sampled: every gradient is written, as zero."""
    case = _case(39, ((7, 9),), 64, 8, anchors=20)
    case[3][...] = 2.0
    grad_out = torch.ones(2, 20, 64)
    assert all((g == 0).all() for g in _backward(case, grad_out))


@gpu
def test_captured_backward_replays():
    """A graph of the backward, replayed on changed inputs, equals the eager call."""
    case = [t.to(DEV) for t in _case(41, ((9, 13), (4, 6)), 256, 8, anchors=60)]
    grad_out = torch.randn(2, 60, 256, generator=torch.Generator().manual_seed(42)).to(DEV)
    lib = load_native_module()
    grads = [torch.empty_like(case[i]) for i in (0, 3, 4)]
    lib.deformable_aggregation_backward(*case, grad_out, *grads)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        lib.deformable_aggregation_backward(*case, grad_out, *grads)
    for step in range(3):
        grad_out.mul_(-0.5)
        case[3].copy_((case[3] + 0.125 * step) % 1.0)
        eager = [torch.empty_like(g) for g in grads]
        lib.deformable_aggregation_backward(*case, grad_out, *eager)
        for g in grads:
            g.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        for g, e in zip(grads, eager):
            torch.testing.assert_close(g, e, rtol=1e-6, atol=1e-6)


@gpu
@pytest.mark.parametrize("offset,short", [(0, 0), (8, 0), (128, 0), (1, 0), (0, 1)])
def test_misaligned_or_short_workspace_is_left_alone(offset, short):
    """A workspace off a 256-byte boundary, or a byte too small, takes the kernels
    without one: right gradients, and not a byte of it written."""
    case = [t.to(DEV) for t in _case(43, ((9, 13), (4, 6)), 256, 8, anchors=60)]
    grad_out = torch.randn(2, 60, 256, generator=torch.Generator().manual_seed(44)).to(DEV)
    lib = load_native_module()
    dims = [2, 3, case[0].shape[1], 256, 2, 60, 3, 8]
    size = lib.raw("deformable_aggregation_backward_workspace_size")(*dims)
    workspace = torch.full((size + 256,), 0x5A, dtype=torch.uint8, device=DEV)
    assert workspace.data_ptr() % 256 == 0
    grads = [torch.full_like(case[i], float("nan")) for i in (0, 3, 4)]
    code = lib.raw("deformable_aggregation_backward_ws")(
        *[t.data_ptr() for t in (*case, grad_out, *grads)], *dims, workspace.data_ptr() + offset,
        size - short, torch.cuda.current_stream().cuda_stream)
    assert code == 0
    assert bool((workspace == 0x5A).all()) == bool(offset or short)
    expected = _backward(case, grad_out)
    for g, e, atol in zip(grads, expected, (1e-5, 1e-3, 1e-4)):
        torch.testing.assert_close(g.cpu(), e, rtol=1e-5, atol=atol)


@gpu
@pytest.mark.parametrize("offset", [0, 1, 2, 3])
@pytest.mark.parametrize("shapes", [((1, 1),), ((3, 5), (2, 2))])
def test_gradient_zeroed_in_full_and_no_further(offset, shapes):
    """Without a workspace the feature gradient is zeroed first, whatever the
    alignment of its ends (3 channels, so its length is no multiple of four)."""
    case = [t.to(DEV) for t in _case(51, shapes, 3, 1, anchors=7, batch=1, cams=1)]
    grad_out = torch.randn(1, 7, 3, generator=torch.Generator().manual_seed(52)).to(DEV)
    n = case[0].numel()
    buffer = torch.full((n + 8,), 7.0, device=DEV)
    rest = [torch.empty_like(case[i]) for i in (3, 4)]
    lib = load_native_module()
    code = lib.raw("deformable_aggregation_backward_ws")(
        *[t.data_ptr() for t in (*case, grad_out)], buffer.data_ptr() + 4 * (offset + 4),
        *[t.data_ptr() for t in rest], *_dims(case), None, 0,
        torch.cuda.current_stream().cuda_stream)
    assert code == 0
    got, outside = buffer[offset + 4: offset + 4 + n], torch.ones(n + 8, dtype=torch.bool)
    outside[offset + 4: offset + 4 + n] = False
    assert (buffer.cpu()[outside] == 7.0).all()
    base = _backward(case, grad_out, "deformable_aggregation_backward_base")
    torch.testing.assert_close(got.cpu().view_as(base[0]), base[0], rtol=1e-5, atol=1e-5)


@gpu
def test_scratch_that_cannot_be_had(monkeypatch):
    """Out of memory for the scratch alone: the call takes the kernels without it."""
    case = _case(45, ((9, 13), (4, 6)), 256, 8, anchors=60)
    grad_out = torch.randn(2, 60, 256, generator=torch.Generator().manual_seed(46))
    expected = _operator_backward(case, grad_out)
    asked, empty = [], torch.empty

    def no_bytes(*args, **kwargs):
        if kwargs.get("dtype") == torch.uint8:
            asked.append(args)
            raise torch.OutOfMemoryError("out of memory")
        return empty(*args, **kwargs)

    monkeypatch.setattr(torch, "empty", no_bytes)
    actual = _operator_backward(case, grad_out)
    assert asked
    for a, e, atol in zip(actual, expected, (1e-5, 1e-3, 1e-4)):
        torch.testing.assert_close(a, e, rtol=1e-5, atol=atol)


def test_workspace_size_and_validation(native_lib):
    size = native_lib.raw("deformable_aggregation_backward_workspace_size")
    dims = [2, 3, 500, 256, 2, 40, 4, 8]  # batch, cams, feat, embeds, scales, anchors, pts, groups
    need = 2 * 3 * 160 * 16 + 2 * 500 * 8 + 4 * 2 * 160 * 3 * 2 * 8
    assert need <= size(*dims) <= need + 5 * 256
    assert size(2, 3, 500, 96, 2, 40, 4, 8) == 0  # no row kernel for 96 channels
    assert size(2, 3, 500, 256, 2, 0, 4, 8) == 0  # nothing sampled
    assert size(2, 3, 500, 256, 2, 40, 4, 9) == 0  # invalid
    assert size(64, 6, 2000, 256, 4, 1 << 20, 8, 8) == 0  # past 32-bit offsets
    fn = native_lib.raw("deformable_aggregation_backward_ws")
    assert fn(*[1] * 5, None, *[1] * 3, *dims, None, 0, None) == 1  # grad_output NULL
    assert "null tensor pointer" in native_lib.last_error()
    assert fn(*[1] * 9, *dims[:7], 9, None, 0, None) == 1
    assert "num_groups must be in [1, 8]" in native_lib.last_error()


@pytest.mark.parametrize("dims,owner", [
    # batch, cams, feat, embeds, scales, anchors, pts, groups
    ([8, 6, 89760, 256, 4, 900, 13, 8], True),    # SparseDrive's batch
    ([1, 1, 500, 128, 2, 50, 5, 8], True),        # the smallest maps and fewest points
    ([1, 1, 500, 64, 2, 50, 5, 8], True),
    ([2, 6, 60000, 128, 1, 1227, 5, 8], False),   # one scale
    ([1, 1, 32768, 256, 2, 900, 13, 8], True),    # 32768 rows a camera ...
    ([1, 1, 32769, 256, 2, 900, 13, 8], False),   # ... more, and one (entry, camera)
    ([4, 1, 50000, 256, 2, 12500, 1, 8], True),   # four of them, and many pairs
    ([4, 1, 50000, 256, 2, 12499, 1, 8], False),
    ([3, 1, 50000, 256, 2, 12500, 1, 8], False),
    ([4, 1, 50000, 64, 2, 12500, 1, 8], False),   # 64 channels
    ([1, 1, 500, 96, 2, 50, 5, 8], False),        # no row kernel
    ([1, 1, 500, 128, 2, 0, 5, 8], False),        # nothing sampled
])
def test_which_shapes_take_the_sums_by_owner(native_lib, dims, owner):
    assert native_lib.raw("deformable_aggregation_backward_prefers_workspace")(*dims) == owner
