"""When the attention backward forms dQ, dK and dV of 16-bit rings in one launch, on the CPU: the library's own rule, for 256 compute units."""

import ctypes
import random

import pytest
import torch

import jigsaw_amd
from jigsaw_amd import _lib

# heads, queries, keys a chunk, head size, chunks: rows of a workgroup of the one launch in bf16 and fp16 (0: two launches)
ONE_LAUNCH = {
    # workgroups of 32, 64 and 128 rows; chunks from 128 keys on and shorter ones
    (10, 22, 130, 32, 1): (32, 32), (3, 24, 89, 24, 2): (32, 32), (68, 80, 141, 32, 1): (64, 64), (79, 37, 29, 8, 4): (64, 64),
    (78, 201, 252, 32, 1): (128, 128), (71, 132, 95, 24, 3): (64, 64), (119, 65, 87, 8, 1): (128, 128),
    (1, 59, 375, 64, 1): (32, 32), (2, 31, 89, 40, 2): (32, 32), (74, 22, 206, 64, 1): (64, 64), (56, 61, 27, 56, 1): (64, 64),
    (55, 203, 194, 64, 1): (0, 128), (57, 139, 88, 64, 2): (64, 64), (91, 71, 72, 56, 1): (128, 128), (100, 71, 154, 56, 1): (128, 128),
    (4, 1, 300, 64, 2): (32, 32), (4, 300, 1, 32, 2): (32, 32),
    # wider heads: the same three, where all workgroups fit at once
    (5, 66, 70, 96, 1): (32, 32), (13, 102, 130, 128, 2): (32, 32), (3, 260, 200, 80, 3): (32, 32), (16, 200, 150, 96, 3): (64, 64),
    (2, 1000, 900, 128, 2): (32, 32), (40, 90, 100, 72, 4): (0, 0), (1, 500, 700, 120, 1): (32, 32), (20, 60, 60, 96, 2): (64, 64),
    (22, 130, 130, 96, 3): (128, 128), (36, 101, 101, 96, 3): (128, 128), (9, 100, 60, 120, 3): (32, 32), (13, 60, 50, 128, 2): (64, 64),
    (8, 333, 333, 128, 3): (64, 64), (32, 204, 204, 128, 2): (128, 128), (28, 70, 70, 128, 4): (128, 128),
}
_TYPES = (torch.bfloat16, torch.float16)


def one_launch_rows(h, sq, sk, d, P, dtype) -> int:
    fn = _lib.load().jg_attn_bwd_one_launch_rows
    fn.restype, fn.argtypes = ctypes.c_int, [ctypes.c_int64] * 5 + [ctypes.c_int]
    return fn(P, h, sq, sk, d, _lib.dtype_code(dtype))


def on_256_compute_units() -> bool:
    return not torch.cuda.is_available() or torch.cuda.get_device_properties(0).multi_processor_count == 256


pytestmark = pytest.mark.skipif(not on_256_compute_units(), reason="the routes are those of 256 compute units")


def test_the_listed_rings_reach_every_kernel():
    reached = set()
    for (h, sq, sk, d, P), rows in ONE_LAUNCH.items():
        assert tuple(one_launch_rows(h, sq, sk, d, P, t) for t in _TYPES) == rows, (h, sq, sk, d, P)
        reached |= {(max(32, -(-d // 32) * 32), t, r, sk < 128) for t, r in zip(_TYPES, rows) if r}
    assert reached == {(d, t, r, short) for d in (32, 64, 96, 128) for t in _TYPES for r in (32, 64, 128) for short in (False, True)}


# heads, tokens, chunks, head size: the rings that the comments beside the rule name
@pytest.mark.parametrize("ring", [
    (4, 128, 2, 32), (15, 710, 3, 32), (3, 1497, 2, 32), (16, 802, 3, 32), (3, 3000, 4, 32), (64, 64, 1, 64), (48, 69, 3, 64), (7, 387, 6, 64),
    (6, 400, 4, 64), (13, 102, 2, 128), (7, 265, 1, 128), (2, 2000, 2, 128), (2, 1000, 3, 96), (16, 200, 3, 96), (40, 90, 4, 80), (1, 2500, 2, 96),
    (28, 205, 3, 96), (9, 235, 5, 80),
])
def test_rings_that_gain_take_one_launch(ring):
    h, n, P, d = ring
    assert all(one_launch_rows(h, n, n, d, P, t) for t in _TYPES)


@pytest.mark.parametrize("ring", [(8, 1024, 8, 32), (24, 1000, 2, 64), (15, 313, 7, 64), (12, 1180, 1, 96), (12, 503, 2, 80), (11, 845, 2, 80), (8, 512, 4, 128),
                                  (33, 193, 3, 128), (30, 140, 4, 128)])
def test_rings_that_the_rule_leaves_take_two(ring):
    h, n, P, d = ring
    assert not any(one_launch_rows(h, n, n, d, P, t) for t in _TYPES)


def test_lengths_in_multiples_of_128_keep_two_launches_at_64_columns_of_bf16():
    for h, n, P in ((4, 128, 2), (4, 512, 4), (8, 256, 2), (1, 1024, 1)):
        assert one_launch_rows(h, n, n, 64, P, torch.bfloat16) == 0 and one_launch_rows(h, n, n, 64, P, torch.float16) != 0


def test_one_launch_has_no_more_workgroups_than_a_grid_holds():
    """Its dQ and dK/dV workgroups lie in one dimension of the grid: 2^32 threads, 256 a workgroup."""
    rng, near, taken = random.Random(5), 0, 0
    cases = [(65535, 64, 1024, 32, 16), (65535, 64, 1024, 8, 16), (65535, 64, 1000, 32, 16), (65535, 128, 1024, 32, 15), (65535, 3, 4096, 24, 8)]
    cases += [(rng.randint(30000, 65535), rng.randint(1, 128), rng.randint(500, 4096), rng.choice((8, 32, 64)), rng.randint(4, 16)) for _ in range(2000)]
    for h, sq, sk, d, P in cases:
        blocks = lambda rows: h * (-(-sq // rows) - P * (-sk // rows))  # noqa: B023, E731
        near += blocks(64) >= 1 << 24
        for t in _TYPES:
            rows = one_launch_rows(h, sq, sk, d, P, t)
            taken += rows != 0
            assert rows == 0 or blocks(rows) < 1 << 24
    assert near > 100 and taken > 100
