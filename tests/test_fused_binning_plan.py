"""Which shapes ms_deform_attn_forward_bin runs as the forward kernel with the
backward's record stores fused in (host-side planning only, no launch).

Every BASELINE training config (c1-c4, fp32 and 16-bit values) writes its
location and weight gradients straight to sample order (slab span at most
8 MB), so both forms are possible there: c2 and the decoder-sized shapes store the
records from the forward kernel, the others run the binning kernels before the
forward that keeps a slab's coarse levels in LDS. A span above 8 MB takes the
records-plus-gather backward and the unfused binning, and channel counts
without a row kernel take the atomic backward (nothing to bin).
"""

import pytest
import torch

from muspace_amd.workloads import CONFIGS


def _meta(cfg, value_dtype, geometry_dtype=torch.float32):
    value = torch.empty((cfg.batch, cfg.spatial_size, cfg.heads, cfg.channels),
                        dtype=value_dtype, device="meta")
    loc = torch.empty((cfg.batch, cfg.queries, cfg.heads, cfg.num_levels, cfg.points, 2),
                      dtype=geometry_dtype, device="meta")
    return value, loc


@pytest.mark.parametrize("name,value_dtype,fused", [
    ("c1", torch.float32, False), ("c2", torch.float32, True), ("c3", torch.float32, False),
    ("c4", torch.bfloat16, False), ("c4", torch.float16, False),
    ("bevformer-1l", torch.float32, False),
])
def test_baseline_training_configs(native_lib, name, value_dtype, fused):
    value, loc = _meta(CONFIGS[name], value_dtype)
    assert native_lib.forward_bin_fuses(value, loc) == fused


@pytest.mark.parametrize("name,value_dtype,geometry_dtype,fused", [
    ("c1", torch.float32, torch.float32, False), ("c2", torch.float32, torch.float32, True),
    ("c4", torch.bfloat16, torch.float32, False),
    # stored 16-bit probabilities would lose the forward precision
    ("c4", torch.bfloat16, torch.bfloat16, True), ("c4", torch.float16, torch.float16, True),
])
def test_softmax_training_configs(native_lib, name, value_dtype, geometry_dtype, fused):
    value, loc = _meta(CONFIGS[name], value_dtype, geometry_dtype)
    assert native_lib.forward_softmax_bin_fuses(value, loc) == fused


@pytest.mark.parametrize("value_dtype,batch,queries,levels,points,fused", [
    (torch.float32, 2, 900, ((100, 167), (50, 84), (25, 42), (13, 21)), 4, True),  # few samples
    (torch.float32, 2, 20000, ((90, 100), (70, 80)), 8, True),   # no level in LDS, full steps
    (torch.float32, 2, 20000, ((90, 100), (70, 80)), 5, False),  # ... ragged ones
    (torch.bfloat16, 2, 20000, ((90, 100), (70, 80)), 5, True),  # 16 bits: not for those
    (torch.float32, 6, 10000, ((116, 200), (58, 100), (29, 50), (15, 25)), 8, True),  # 32 samples
    (torch.bfloat16, 6, 10000, ((116, 200), (58, 100), (29, 50), (15, 25)), 8, False),
    (torch.float32, 1, 8162, ((46, 81), (23, 41), (12, 21), (6, 11), (3, 6)), 5, False),
    (torch.float32, 2, 40000, ((200, 200),), 4, False),  # one level: 128 chunks
    (torch.float32, 4, 40000, ((200, 200),), 4, True),   # ... 64
    (torch.float16, 2, 40000, ((100, 100),), 4, True),
])
def test_which_form_bins(native_lib, value_dtype, batch, queries, levels, points, fused):
    value = torch.empty((batch, sum(h * w for h, w in levels), 8, 32), dtype=value_dtype,
                        device="meta")
    loc = torch.empty((batch, queries, 8, len(levels), points, 2), device="meta")
    assert native_lib.forward_bin_fuses(value, loc) == fused


def test_span_above_8mb_takes_the_binning_kernels(native_lib):
    # one slab of 22000 queries x 32 samples x 12 bytes = 8.4 MB
    value = torch.empty((1, 600, 2, 32), device="meta")
    loc = torch.empty((1, 22000, 2, 1, 32, 2), device="meta")
    assert not native_lib.forward_bin_fuses(value, loc)
    small = torch.empty((1, 10000, 2, 1, 32, 2), device="meta")
    assert native_lib.forward_bin_fuses(value, small)


@pytest.mark.parametrize("channels", [3, 8, 12])
def test_channels_without_a_tile_path_do_not_fuse(native_lib, channels):
    value = torch.empty((2, 300, 4, channels), device="meta")
    loc = torch.empty((2, 200, 4, 2, 4, 2), device="meta")
    assert not native_lib.forward_bin_fuses(value, loc)


@pytest.mark.parametrize("cells,queries,levels,points,binned", [
    (192959, 100, 3, 4, True),   # 14843 tiles of 13 cells, and one a level and one more
    (192985, 100, 3, 4, False),  # 14845, so past 14847 with those
    (4000, 100, 1, 2048, True),  # 2048 sample slots a query
    (4000, 100, 1, 2049, False),
])
def test_limits_of_the_binned_backward(native_lib, cells, queries, levels, points, binned):
    value = torch.empty((1, cells, 1, 32), device="meta")
    loc = torch.empty((1, queries, 1, levels, points, 2), device="meta")
    assert (native_lib.backward_workspace_bytes(value, loc) > 0) == binned
