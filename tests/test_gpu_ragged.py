"""Sizes at the edges of the kernels' tiles: short, odd and unaligned rows,
small planes, one-row and many-row reductions."""
import ctypes as C
import zlib

import numpy as np
import pytest

import oracle
from gpu_helpers import (_offset_dev, batchnorm_bwd, batchnorm_fwd, binary_bwd, binary_fwd, gemm,
                         layernorm_bwd, layernorm_fwd, reduce, rng_normal, rng_uniform)

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


# One size per form of the small-tile product (16- and 32-wide tiles with k
# over 4 or 16 waves, 64-wide tiles) and its edges: a partial step only, one
# full step and a rest, fewer steps than waves, rows past a tile, odd leading
# dimensions, more problems than one.
SMALL_PRODUCTS = [(1, 1, 1, 1), (3, 17, 33, 5), (16, 16, 31, 1), (65, 128, 130, 1), (16, 512, 333, 1), (1, 70, 4100, 1),
                  (300, 10, 768, 1), (33, 47, 8200, 1), (40, 3000, 65, 1), (700, 900, 30, 1), (1500, 1201, 97, 1),
                  (2, 64, 333, 24)]


@pytest.mark.parametrize("m,n,k,batch", SMALL_PRODUCTS)
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_small_products(wm, m, n, k, batch, ta, tb):
    """alpha, accumulation and bias, leading dimensions 1 and 3 past a row
    (NaN there), against float64 within 1e-5 of the sum of |terms|."""
    r = np.random.default_rng(seed_of(m, n, k, ta, tb))
    a, b = r.standard_normal((batch, m, k), np.float32), r.standard_normal((batch, k, n), np.float32)
    lda, ldb, ldc = (m if ta else k) + 1, (k if tb else n) + 3, n + 1

    def stored(x, trans, ld):
        s = x.transpose(0, 2, 1) if trans else x
        buf = np.full(s.shape[:2] + (ld,), np.nan, np.float32)
        buf[..., :s.shape[2]] = s
        return buf

    sa, sb = stored(a, ta, lda), stored(b, tb, ldb)
    c0 = r.standard_normal((batch, m, ldc), np.float32)
    bias = r.standard_normal(n, np.float32)
    st = (sa[0].size, 0, sb[0].size, 0, c0[0].size, 0)
    ref = np.matmul(a.astype(np.float64), b)
    scale = np.matmul(np.abs(a).astype(np.float64), np.abs(b))
    for acc, bi in ((0, None), (1, None), (0, bias), (1, bias)):
        got = gemm(ta, tb, m, n, k, 0.5, sa.ravel(), lda, sb.ravel(), ldb, c0.ravel(), ldc, acc, bi, batch, 1, st)
        got = got.reshape(c0.shape)
        add = (c0[..., :n] if acc else 0.0) + (bias if bi is not None else 0.0)
        size = (np.abs(c0[..., :n]) if acc else 0.0) + (np.abs(bias) if bi is not None else 0.0)
        ok, w = oracle.close_scaled(got[..., :n], 0.5 * ref + add, 0.5 * scale + size, RTOL)
        assert ok, f"{w:.3g}x tolerance"
        assert np.array_equal(got[..., n:], c0[..., n:])  # past the rows: untouched


# Weight gradients x^T dY on the k split of the direct-to-LDS kernel (with the library
# route off; by default the library keeps some): 18 and 200 tiles, equal slices and
# a shorter last one, and sizes next to those.
@pytest.mark.parametrize("m,n,k", [(384, 768, 4096), (768, 384, 4160), (640, 512, 6848), (2560, 1280, 4096),
                                   (384, 768, 4032), (128, 2176, 4096), (1024, 1024, 4096), (384, 768, 4100)])
@pytest.mark.parametrize("route", [0, 1])
def test_long_weight_gradients(wm, m, n, k, route):
    """alpha and accumulation, rows 4 past their end (NaN there), against float64
    within 1e-5 of the sum of |terms|; the same bits again."""
    r = np.random.default_rng(seed_of(m, n, k))
    x, dy = np.full((k, m + 4), np.nan, np.float32), np.full((k, n + 4), np.nan, np.float32)
    x[:, :m], dy[:, :n] = r.standard_normal((k, m), np.float32), r.standard_normal((k, n), np.float32)
    c0 = r.standard_normal((m, n + 4), np.float32)
    ref = x[:, :m].T.astype(np.float64) @ dy[:, :n]
    scale = np.abs(x[:, :m].T).astype(np.float64) @ np.abs(dy[:, :n])
    old = wm.lib().wm_gemm_library(-1)
    wm.lib().wm_gemm_library(route)
    try:
        for acc in (0, 1):
            got = [gemm(1, 0, m, n, k, 0.5, x.ravel(), m + 4, dy.ravel(), n + 4, c0.ravel(), n + 4, acc, None, 1, 1,
                        None).reshape(c0.shape) for _ in range(2)]
            base = c0[:, :n] if acc else 0.0
            ok, w = oracle.close_scaled(got[0][:, :n], 0.5 * ref + base, 0.5 * scale + np.abs(base), RTOL)
            assert ok, f"{w:.3g}x tolerance"
            assert np.array_equal(got[0], got[1])
            assert np.array_equal(got[0][:, n:], c0[:, n:])
    finally:
        wm.lib().wm_gemm_library(old)


# Both sides of each line between the k split and the library (which launches no
# kernel of this library).
@pytest.mark.parametrize("m,n,k,split", [
    (768, 384, 3072, True), (768, 384, 3008, False), (384, 768, 3072, False), (2176, 128, 3072, False),
    (384, 1408, 3072, True), (256, 2048, 3072, False), (512, 1536, 3072, True), (896, 896, 3072, True),
    (896, 1024, 3072, False), (1024, 1024, 3072, False), (640, 1664, 3072, True), (640, 2048, 3072, True),
    (768, 1792, 3072, False), (640, 3328, 3072, True), (1024, 2176, 3072, False), (2432, 1280, 3072, True),
    (3072, 1024, 3072, False), (1664, 1920, 3072, False), (2560, 1280, 3072, False)])
def test_weight_gradient_route_lines(wm, m, n, k, split):
    """Whole numbers: exact in float32 in any order."""
    r = np.random.default_rng(seed_of("route", m, n, k))
    x, dy = (r.integers(-3, 4, (k, w)).astype(np.float32) for w in (m, n))
    before, after = C.c_int64(), C.c_int64()
    wm.call("wm_launch_count", C.byref(before))
    got = gemm(1, 0, m, n, k, 1.0, x.ravel(), m, dy.ravel(), n, np.zeros(m * n, np.float32), n, 0, None, 1, 1, None)
    wm.call("wm_launch_count", C.byref(after))
    assert (after.value > before.value) == split
    assert np.array_equal(got.reshape(m, n), (x.T.astype(np.float64) @ dy).astype(np.float32))


@pytest.mark.parametrize("offset", [0, 1, 2])
@pytest.mark.parametrize("rows,cols", [(1, 1), (5, 3), (7, 4), (600, 13), (3, 127), (300, 255), (5, 1023), (4, 1024),
                                       (3, 1025), (2, 4099), (3, 32772), (2, 33001)])
def test_cross_entropy_rows_at_any_alignment(wm, rows, cols, offset):
    """Logits and gradient starting `offset` floats past a 16-byte boundary:
    loss and gradient (written, then accumulated) within 1e-5 of the fp64
    oracle's scale, and nothing written before or after the gradient."""
    s = seed_of("ce", rows, cols)
    x = rng_normal((rows, cols), s, 3.0)
    x[0, cols // 2] = 40.0
    if cols > 4:
        x[-1, :cols // 3] = -np.inf
    lab = (np.arange(rows) * 7 + cols - 1) % cols
    lab[-1] = cols - 1  # a -inf label entry would make the loss infinite, with nothing left to compare
    dx, px = _offset_dev(x, offset)
    dl, dg = wm.DeviceArray.from_host(lab.astype(np.float32)), wm.DeviceArray.from_host(np.float32([0.75]))
    stats, loss = wm.DeviceArray((rows, wm.CE_STATS)), wm.DeviceArray((1,))
    wm.call("wm_cross_entropy_fwd", px, dl.vp, rows, cols, stats.vp, loss.vp)
    ref = oracle.get("f64").cross_entropy(x, lab.astype(np.float32))
    assert abs(loss.to_host()[0] - ref) <= RTOL * max(abs(ref), 1.0)
    buf = rng_normal((offset + rows * cols + 8,), s + 1)
    gx = wm.DeviceArray.from_host(buf)
    pg = C.c_void_p(gx.ptr + 4 * offset)
    r64 = oracle.get("f64").cross_entropy_bwd(x, lab.astype(np.float32), 0.75)
    scale = oracle.get("abs").cross_entropy_bwd(x, lab.astype(np.float32), 0.75)
    for acc in (1, 0):
        wm.call("wm_cross_entropy_bwd", px, dl.vp, stats.vp, dg.vp, pg, acc, rows, cols)
        got = gx.to_host()
        g = got[offset:offset + rows * cols].reshape(rows, cols)
        g0 = buf[offset:offset + rows * cols].reshape(rows, cols) if acc else np.zeros((rows, cols), np.float32)
        ok, w = oracle.close_scaled(g, r64 + g0, scale + np.abs(g0), RTOL, 1e-30)
        assert ok, f"{w:.3g}x tolerance (accumulate {acc})"
        assert np.array_equal(got[:offset], buf[:offset])
        assert np.array_equal(got[offset + rows * cols:], buf[offset + rows * cols:])


# Channels at the ends of each register tile (256 or 1024 threads, 1 to 4
# float4s or 8 floats each) and just past the largest, planes of one float,
# of less than a wave and across workgroup steps.
@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("shape", [(1, 2, 1, 1), (255, 2, 1, 1), (257, 3, 1, 1), (64, 5, 2, 2), (4, 3, 32, 32),
                                   (4, 3, 36, 32), (16, 2, 32, 32), (17, 2, 32, 32), (91, 3, 9, 10), (92, 3, 9, 10),
                                   (200, 2, 7, 7), (40, 70, 14, 14), (3, 2, 200, 100)])
def test_batchnorm_channel_sizes(wm, shape, accumulate):
    s = seed_of("bn", shape)
    o64, oab, ch = oracle.get("f64"), oracle.get("abs"), shape[1]
    x, g = rng_normal(shape, s) + np.float32(0.5), rng_normal(shape, s + 1)
    gamma, beta = rng_uniform((ch,), s + 2, 0.5, 1.5), rng_normal((ch,), s + 3)
    rm, rv = rng_normal((ch,), s + 4), rng_uniform((ch,), s + 5, 0.5, 1.5)
    y, mean, inv, rm1, rv1 = batchnorm_fwd(x, gamma, beta, rm, rv, True)
    y64, m64, i64, rm64, rv64 = o64.batchnorm2d(x, gamma, beta, rm, rv, training=True)
    xs = np.abs(x).mean((0, 2, 3))
    for got, ref, scale in ((y, y64, oab.batchnorm2d(x, gamma, beta, rm, rv, training=True)[0]), (mean, m64, xs),
                            (inv, i64, i64), (rm1, rm64, 0.9 * np.abs(rm) + 0.1 * xs), (rv1, rv64, rv64)):
        ok, w = oracle.close_scaled(got, ref, scale, RTOL, 1e-30)
        assert ok, f"forward {w:.3g}x tolerance"
    g0 = (rng_normal(shape, s + 6), rng_normal((ch,), s + 7), rng_normal((ch,), s + 8)) if accumulate else (None,) * 3
    got = batchnorm_bwd(g, x, gamma, mean, inv, *g0)
    ref, scale = o64.batchnorm2d_bwd(g, x, gamma, mean, inv), oab.batchnorm2d_bwd(g, x, gamma, mean, inv)
    for k in range(3):
        z = g0[k] if accumulate else np.float32(0)
        ok, w = oracle.close_scaled(got[k], ref[k] + z, scale[k] + np.abs(z), RTOL, 1e-30)
        assert ok, f"gradient {k} {w:.3g}x tolerance"


# Rows at the ends of each LayerNorm tile (1 to 4 float4s of a wave, 256 and
# 1024 threads), odd lengths, and few or many rows per workgroup.
@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("rows,n", [(1, 1), (3, 7), (35, 74), (9, 256), (5, 257), (1100, 512), (33, 768), (300, 767),
                                    (2100, 1024), (7, 1025), (12, 2048), (5, 2052), (9, 4100), (10, 8192)])
def test_layernorm_row_lengths(wm, rows, n, accumulate):
    s = seed_of("ln", rows, n)
    o64, oab = oracle.get("f64"), oracle.get("abs")
    x, g = rng_normal((rows, n), s), rng_normal((rows, n), s + 1)
    gamma, beta = rng_uniform((n,), s + 2, 0.5, 1.5), rng_normal((n,), s + 3)
    y, mean, inv = layernorm_fwd(x, gamma, beta)
    ok, w = oracle.close_scaled(y, o64.layernorm(x, gamma, beta)[0], oab.layernorm(x, gamma, beta)[0], RTOL, 1e-30)
    assert ok, f"forward {w:.3g}x tolerance"
    g0 = (rng_normal((rows, n), s + 4), rng_normal((n,), s + 5), rng_normal((n,), s + 6)) if accumulate else (None,) * 3
    got = layernorm_bwd(g, x, gamma, mean, inv, *g0)
    ref, scale = o64.layernorm_bwd(g, x, gamma, mean, inv), oab.layernorm_bwd(g, x, gamma, mean, inv)
    for k in range(3):
        z = g0[k] if accumulate else np.float32(0)
        ok, w = oracle.close_scaled(got[k], ref[k] + z, scale[k] + np.abs(z), RTOL, 1e-30)
        assert ok, f"gradient {k} {w:.3g}x tolerance"


# Strided reductions at the ends of the one-dispatch range (sixteen waves on up
# to 320 or 512 positions) and just past it, below one position per wave, in
# part-filled tiles of floats and float4s.
@pytest.mark.parametrize("outer,n,inner", [(1, 129, 4), (1, 320, 10), (1, 321, 10), (3, 200, 64), (2, 130, 257),
                                           (64, 197, 768), (140, 512, 3), (140, 513, 3), (130, 300, 36)])
def test_strided_reductions_short_axis(wm, outer, n, inner):
    x = np.rint(rng_normal((outer, n, inner), seed_of("red", outer, n, inner)) * 8).astype(np.float32) / 8  # ties
    x[0, 0, 0] = np.nan  # a NaN wins only as the first element
    x[0, n // 2, 1] = np.nan
    x[-1, :, -1] = -np.inf
    for op in ("max", "min", "argmax", "sum", "mean"):
        y = np.nan_to_num(x, neginf=0.0) if op in ("sum", "mean") else x
        v, i = reduce(op, y, outer, n, inner, want_idx=op in ("max", "min"))
        if op in ("sum", "mean"):
            ref, scale = (oracle.get(k).reduce(op, y, outer, n, inner)[0] for k in ("f64", "abs"))
            ok, w = oracle.close_scaled(v, ref, scale, RTOL, 1e-30)
            assert ok, f"{op} {w:.3g}x tolerance"
        else:
            rv, ri = oracle.get("f32").reduce(op, y, outer, n, inner)
            assert oracle.bit_equal(v, rv), op
            assert i is None or np.array_equal(i, ri), op


# The lines between sixteen waves on the whole axis and chunks of it: 160 and 256
# positions of few float4 tiles, 512 of 192 tiles (3/4 of the CUs), of 256 float tiles.
@pytest.mark.parametrize("outer,n,inner", [(1, 160, 64), (1, 161, 64), (2, 256, 256), (2, 257, 256), (191, 300, 4),
                                           (192, 300, 4), (192, 513, 4), (256, 512, 3), (257, 512, 3)])
def test_strided_reductions_route_lines(wm, outer, n, inner):
    test_strided_reductions_short_axis(wm, outer, n, inner)


# Broadcast forwards over rows of whole float4s that are not whole tiles, the
# broadcast operand along the row, along the outer dims and both.
@pytest.mark.parametrize("op", ["add", "div", "max"])
@pytest.mark.parametrize("full,vec", [((5, 4), (5, 1)), ((3, 7, 12), (7, 1)), ((6, 5, 36), (1, 5, 1)), ((700, 64), (64,)),
                                      ((9, 768), (9, 1)), ((2, 3, 5, 196), (3, 1, 196)), ((4, 6, 3136), (1, 6, 1)),
                                      ((3, 2, 4, 2, 8), (2, 1, 2, 1)), ((2, 900), (1, 900)), ((33, 1028), (33, 1))])
def test_broadcast_forward_ragged_rows(wm, op, full, vec):
    s = seed_of(op, full, vec)
    a, b = rng_normal(full, s), rng_uniform(vec, s + 1, 0.5, 2.0)
    for x, y in ((a, b), (b, a)):
        assert oracle.bit_equal(binary_fwd(op, x, y), oracle.get("f32").binary(op, x, y))
    c, d = rng_normal(full[:-1] + (1,), s + 2), rng_uniform(full[-1:], s + 3, 0.5, 2.0)
    assert oracle.bit_equal(binary_fwd(op, c, d), oracle.get("f32").binary(op, c, d))


# Column sums of row vectors at the lines of their second pass: 4 and 64
# columns per workgroup, a thread per column, and a partial last tile.
@pytest.mark.parametrize("rows,cols", [(37, 2044), (37, 2048), (9, 16380), (9, 16384), (3, 65532), (5, 65536),
                                       (70, 65540), (2, 300004)])
@pytest.mark.parametrize("accumulate", [False, True])
def test_wide_row_vector_gradient(wm, rows, cols, accumulate):
    """Small whole numbers: every sum is exact in float32."""
    r = np.random.default_rng(seed_of("wide", rows, cols))
    g = r.integers(-8, 9, (rows, cols)).astype(np.float32)
    a, b = np.ones((rows, cols), np.float32), np.ones((cols,), np.float32)
    b0 = r.integers(-8, 9, (cols,)).astype(np.float32) if accumulate else None
    ga, gb = binary_bwd("add", g, a, b, None, None, b0)
    assert np.array_equal(ga, g)
    assert np.array_equal(gb, g.sum(0) + (b0 if accumulate else 0.0))


# Many [R, C] problems sharing workgroups: rows of one unit up to more than a
# wave, one to a few rows each (a row lane per row, and several rows per lane
# where there is enough work), a partial last group of problems, more groups
# than a grid's z, and few long rows (tiles of 128 and 256 units).
MANY_SHAPES = [((3, 2, 1), (3, 1, 1)), ((300, 2, 8), (300, 1, 8)), ((70, 3, 7), (70, 1, 7)), ((1001, 5, 4), (1001, 1, 4)),
               ((130, 2, 130), (130, 1, 130)), ((9000, 3, 33), (9000, 1, 33)), ((70000, 2, 3), (70000, 1, 3)),
               ((33, 6, 260), (33, 1, 260)), ((2, 300001), (300001,)), ((3, 4098), (4098,)), ((90, 9, 3, 64), (90, 1, 3, 64))]


@pytest.mark.parametrize("op", ["add", "div", "pow"])
@pytest.mark.parametrize("full,vec", MANY_SHAPES)
def test_broadcast_backward_many_small_problems(wm, op, full, vec):
    test_broadcast_backward_edges(wm, op, full, vec)


# Many channels of a few elements sharing workgroups: planes of 1 to 32 units
# (the longest whose channels share them) and one more, of floats and of
# float4s, one and several row groups, a partial last tile; just fewer channels
# than share them.
CHANNEL_SHAPES = [((2, 4096, 4), (4096, 1)), ((3, 4099, 3), (4099, 1)), ((2, 4100, 31), (4100, 1)),
                  ((3, 4096, 32), (4096, 1)), ((2, 4097, 33), (4097, 1)), ((2, 4098, 128), (4098, 1)),
                  ((2, 4098, 132), (4098, 1)), ((70, 4096, 2), (4096, 1)), ((9, 5000, 4, 4), (5000, 1, 1)),
                  ((300, 4101, 1, 2), (4101, 1, 1)), ((3, 4095, 3), (4095, 1))]


@pytest.mark.parametrize("op", ["add", "div", "pow"])
@pytest.mark.parametrize("full,vec", CHANNEL_SHAPES)
def test_broadcast_backward_many_channels(wm, op, full, vec):
    test_broadcast_backward_edges(wm, op, full, vec)


def test_broadcast_backward_channel_count(wm):
    """More channels than a workgroup each could be launched for (2^32 threads):
    ones, so every channel's sum is its element count."""
    k = (1 << 24) + 3
    full, vec = (2, k, 2), (k, 1)
    g, a, b = (wm.DeviceArray(s) for s in (full, full, vec))
    ga, gb = wm.DeviceArray(full), wm.DeviceArray(vec)
    for d in (g, a, b):
        d.fill(1.0)
    ga.fill(np.nan)
    gb.fill(np.nan)
    wm.binary_bwd(wm.ADD, g, a, b, None, ga, False, gb, False)
    assert np.all(gb.to_host() == 2.0 * full[2])
    assert np.all(ga.to_host() == 1.0)


def kernel_ms(wm, call, reps=12):
    """The kernels' time of one call, the least of `reps`."""
    best = C.c_float()
    ms = []
    for _ in range(reps):
        wm.call("wm_span_begin")
        call()
        wm.call("wm_span_end", C.byref(best), None, None)
        ms.append(best.value)
    return min(ms)


def pace(wm, nbytes, call):
    """How many times longer than a copy of `nbytes` (read and written) a call
    takes."""
    n = nbytes // 32 * 4
    src, dst = wm.DeviceArray((n,)), wm.DeviceArray((n,))
    src.fill(1.0)
    return kernel_ms(wm, call) / kernel_ms(wm, lambda: wm.call("wm_copy_kernel", dst.vp, src.vp, n))


def backward_pace(wm, full, vec):
    """pace() of the add backward of two device tensors of ones."""
    g, a, b = (wm.DeviceArray(s) for s in (full, full, vec))
    ga, gb = wm.DeviceArray(full), wm.DeviceArray(vec)
    for d in (g, a, b):
        d.fill(1.0)
    return pace(wm, 8 * g.size + 4 * b.size, lambda: wm.binary_bwd(wm.ADD, g, a, b, None, ga, False, gb, False))


# A workgroup per problem or channel took 21 to 142 times a copy over these, a
# row vector over two long rows 6.7.
@pytest.mark.parametrize("full,vec", [((1 << 20, 2, 4), (1 << 20, 1, 4)), ((65536, 3, 7), (65536, 1, 7)),
                                      ((2, 4000001), (1, 4000001)), ((2, 1 << 20, 2), (1, 1 << 20, 1)),
                                      ((4, 200000, 3), (1, 200000, 1))])
def test_broadcast_backward_pace(wm, full, vec):
    assert backward_pace(wm, full, vec) < 5.0


def test_layernorm_backward_pace(wm):
    """Wide rows over few enough workgroups that their partials are a small part
    of the traffic (1.13 times a copy; eight workgroups per CU: 1.40)."""
    rows, n = 16384, 2048
    g, x, gx = (wm.DeviceArray((rows, n)) for _ in range(3))
    gamma, dg, db = (wm.DeviceArray((n,)) for _ in range(3))
    mean, inv = wm.DeviceArray((rows,)), wm.DeviceArray((rows,))
    for d in (g, x, gamma, mean, inv):
        d.fill(1.0)
    assert pace(wm, 12 * rows * n, lambda: wm.call("wm_layernorm_bwd", g.vp, x.vp, gamma.vp, mean.vp, inv.vp, rows, n,
                                                   gx.vp, 0, dg.vp, 0, db.vp, 0)) < 1.27


@pytest.mark.parametrize("offset", [0, 3])
@pytest.mark.parametrize("rows,cols", [(3, 5), (3, 6), (70, 17), (130, 20), (130, 21), (9, 159), (9, 161), (7, 319),
                                       (7, 321), (5, 1020), (5, 1021), (3, 1499), (3, 1502), (3, 1503), (3, 1507)])
def test_cross_entropy_rows_a_little_longer_than_their_lanes(wm, rows, cols, offset):
    """Rows whose lanes or tile take a second float4, at the ends of each."""
    test_cross_entropy_rows_at_any_alignment(wm, rows, cols, offset)


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("rows,cols", [(3, 254), (3, 255), (3, 256), (3, 257), (4, 512), (4, 513), (3, 767), (3, 768),
                                       (3, 769), (2049, 257), (6144, 257), (6145, 257), (6145, 255)])
def test_cross_entropy_rows_of_single_floats(wm, rows, cols, offset):
    """Both sides of the widths and row counts between which a written gradient
    takes a workgroup per row, and rows past its grid."""
    test_cross_entropy_rows_at_any_alignment(wm, rows, cols, offset)


@pytest.mark.parametrize("rows,cols", [(511, 255), (512, 254), (512, 255), (512, 257), (2100, 1023), (513, 4099),
                                       (9216, 1021), (9300, 1021)])
def test_nll_backward_rows_of_single_floats(wm, rows, cols):
    """Both sides of the lines between which a workgroup per row writes the
    one-hot gradient; nothing written past its end."""
    lab = ((np.arange(rows) * 7 + cols - 1) % cols).astype(np.float32)
    dl, dg = wm.DeviceArray.from_host(lab), wm.DeviceArray.from_host(np.float32([0.75]))
    buf = rng_normal((rows * cols + 8,), seed_of("nll", rows, cols))
    gx = wm.DeviceArray.from_host(buf)
    wm.call("wm_nll_bwd", dl.vp, dg.vp, gx.vp, 0, rows, cols)
    got = gx.to_host()
    assert oracle.bit_equal(got[:rows * cols].reshape(rows, cols), oracle.get("f32").nll_bwd((rows, cols), lab, 0.75))
    assert np.array_equal(got[rows * cols:], buf[rows * cols:])


def test_cross_entropy_backward_pace(wm):
    """Rows of one float4 more than a workgroup's lanes at some shifts: 1.5 times a
    copy (2.5 with a tile of its own for it)."""
    rows, cols = 32768, 1023
    x, gx = wm.DeviceArray((rows, cols)), wm.DeviceArray((rows, cols))
    lab, g = wm.DeviceArray((rows,)), wm.DeviceArray((1,))
    stats, loss = wm.DeviceArray((rows, wm.CE_STATS)), wm.DeviceArray((1,))
    for d in (x, lab, g):
        d.fill(1.0)
    wm.call("wm_cross_entropy_fwd", x.vp, lab.vp, rows, cols, stats.vp, loss.vp)
    p = pace(wm, 8 * rows * cols, lambda: wm.call("wm_cross_entropy_bwd", x.vp, lab.vp, stats.vp, g.vp, gx.vp, 0, rows,
                                                  cols))
    assert p < 1.95
