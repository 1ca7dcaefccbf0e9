"""Sizes at the edges of the kernels' tiles: short, odd and unaligned rows,
small planes, one-row and many-row reductions."""
import zlib

import numpy as np
import pytest

import oracle
from tests.gpu_helpers import binary_bwd, binary_fwd, rng_normal, rng_uniform

pytestmark = pytest.mark.gpu
RTOL = 1e-5


def seed_of(*key):
    return zlib.crc32(repr(key).encode()) & 0xFFFF


# Column layouts [O, R, C] with [O, 1, C] (row groups of one and of many, 1 to
# 64-unit tiles and a partial one, float and float4 units), channel layouts
# [O, K, I] with [1, K, 1] (one and several chunks, planes below and above a
# workgroup), and same-shape tensors with a tail.
BWD_SHAPES = [
    ((3, 1), (3, 1)), ((7, 5), (7, 5)), ((1, 4099), (1, 4099)),
    ((2, 10), (10,)), ((1500, 10), (10,)), ((17, 64), (64,)), ((300, 768), (768,)), ((70, 257), (257,)),
    ((4200, 3), (1, 3)), ((5, 9, 36), (5, 1, 36)), ((3, 700, 65), (3, 1, 65)), ((2, 33, 1, 130), (2, 1, 1, 130)),
    ((3, 5, 2, 2), (1, 5, 1, 1)), ((4, 3, 7, 7), (3, 1, 1)), ((2, 6, 33, 31), (1, 6, 1, 1)),
    ((9, 2, 64, 64), (1, 2, 1, 1)), ((600, 3, 5), (1, 3, 1)),
]


@pytest.mark.parametrize("op", ["add", "div", "pow"])
@pytest.mark.parametrize("full,vec", BWD_SHAPES)
def test_broadcast_backward_edges(wm, op, full, vec):
    """Both operand orders, overwriting and accumulating, against the fp64
    oracle within 1e-5 of the sum of |terms|."""
    for swap in (False, True):
        sa, sb = (vec, full) if swap else (full, vec)
        s = seed_of(op, sa, sb)
        a = np.abs(rng_normal(sa, s)) + np.float32(0.25)
        b = rng_uniform(sb, s + 1, 0.5, 2.0)
        out = binary_fwd(op, a, b)
        g = rng_normal(out.shape, s + 2)
        ra, rb = oracle.get("f64").binary_bwd(op, g, a, b, out)
        ta, tb = oracle.get("abs").binary_bwd(op, g, a, b, out)
        for acc in (False, True):
            a0 = rng_normal(sa, s + 3) if acc else None
            b0 = rng_normal(sb, s + 4) if acc else None
            ga, gb = binary_bwd(op, g, a, b, out, a0, b0)
            za, zb = (a0, b0) if acc else (0.0, 0.0)
            ok, w = oracle.close_scaled(ga, ra + za, ta + np.abs(za), RTOL)
            assert ok, f"grad a off by {w:.3g}x tolerance (swap {swap}, accumulate {acc})"
            ok, w = oracle.close_scaled(gb, rb + zb, tb + np.abs(zb), RTOL)
            assert ok, f"grad b off by {w:.3g}x tolerance (swap {swap}, accumulate {acc})"
