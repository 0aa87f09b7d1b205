"""Which calls take the forward that keeps a slab's coarse levels in LDS (host-side
planning only, no launch): both sides of every rule of the dispatch.
"""

import pytest
import torch

F32, F16, BF16 = torch.float32, torch.float16, torch.bfloat16


def _takes(lib, vdt, batch, queries, levels, points, heads=8, channels=32, cams=0):
    value = torch.empty((batch, sum(h * w for h, w in levels), heads, channels), dtype=vdt,
                        device="meta")
    loc = torch.empty((batch, queries, heads, len(levels), points, 2), device="meta")
    return lib.forward_takes_slab(value, loc, cams)


SCA = ((116, 200), (58, 100), (29, 50), (15, 25))
DETR = ((100, 167), (50, 84), (25, 42), (13, 21))
ODD = ((75, 101), (38, 51), (19, 26))
TWO = ((200, 200), (100, 100))
SMALL = ((36, 30), (18, 15), (9, 8), (5, 4))


@pytest.mark.parametrize("vdt,batch,queries,levels,points,slab", [
    (F32, 6, 10000, SCA, 8, True),
    (BF16, 6, 10000, SCA, 8, True),
    (F32, 2, 22223, DETR, 4, True),
    (F16, 3, 10007, ODD, 4, True),
    (F32, 1, 1000, ((32, 32), (16, 16), (8, 8), (4, 4)), 4, False),  # few samples
    (F32, 1, 4064, SMALL, 8, False),   # 127 queries of 32 samples a chunk ...
    (F32, 1, 4096, SMALL, 8, True),    # ... 128 of them, two whole rounds
    (F32, 1, 4128, SMALL, 8, False),   # the third round holds one query of 64
    (F32, 1, 4700, SMALL, 8, True),
    (F16, 1, 4096, SMALL, 8, True),    # 16 bits: a round is 128 queries
    (F16, 1, 6900, SMALL, 8, False),   # 216 of 256
    (F16, 1, 7100, SMALL, 8, True),    # 222
    (F32, 2, 20000, TWO, 4, True),     # no level in LDS, and a slab past the L2: 32 chunks
    (F32, 3, 28733, TWO, 4, True),
    (BF16, 2, 20000, TWO, 4, True),    # 16 chunks
    (BF16, 3, 28733, TWO, 4, False),   # 21 chunks of a slab past the L2
    (BF16, 3, 28733, ((80, 110), (40, 55)), 4, True),   # of 1.4 MB of lines
    (BF16, 1, 15400, SCA, 8, True),    # 32 chunks: an XCD a head, 3.9 MB of lines
    (BF16, 1, 15400, TWO, 8, False),   # 6.4 MB
])
def test_levels(native_lib, vdt, batch, queries, levels, points, slab):
    assert _takes(native_lib, vdt, batch, queries, levels, points) == slab


@pytest.mark.parametrize("vdt,batch,queries,levels,points,slab", [
    (F32, 2, 40000, ((200, 200),), 4, True),
    (F32, 2, 32640, ((200, 200),), 4, False),    # 1020 samples a chunk
    (F32, 4, 40000, ((200, 200),), 4, True),     # 64 chunks
    (F32, 5, 40000, ((200, 200),), 4, False),    # 51 chunks of a slab past the L2
    (F32, 5, 40000, ((150, 150),), 4, True),
    (F32, 2, 70000, ((200, 200),), 3, False),    # fewer than four samples
])
def test_one_level(native_lib, vdt, batch, queries, levels, points, slab):
    assert _takes(native_lib, vdt, batch, queries, levels, points) == slab


@pytest.mark.parametrize("vdt,queries,levels,points,slab", [
    (F32, 10000, SCA, 8, True),
    (BF16, 10000, SCA, 8, True),
    (F32, 10000, TWO, 8, False),                      # no level in LDS
    (F32, 10000, (*TWO, (50, 50)), 8, True),          # but ragged steps: 24 samples of 32
    (F32, 10000, ((200, 200),), 8, False),            # one level
    (BF16, 40000, ((60, 70),), 8, False),
    (BF16, 5700, SCA, 8, False),                      # 179 of 256 queries a chunk
    (BF16, 5900, SCA, 8, True),                       # 185
    (BF16, 10000, TWO, 8, False),
])
def test_cameras(native_lib, vdt, queries, levels, points, slab):
    assert _takes(native_lib, vdt, 1, queries, levels, points, cams=6) == slab


@pytest.mark.parametrize("channels", [16, 24, 128])
def test_other_channel_counts(native_lib, channels):
    assert not _takes(native_lib, F32, 6, 10000, SCA, 8, channels=channels)
