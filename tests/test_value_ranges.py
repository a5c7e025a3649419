"""Products and convolutions over the whole range of fp32 values.

An fp32 product rounds each term once: a small element beside a large one
keeps its 24 bits, and a product with one nonzero term is that term. Kernels
that cut their operands into 16-bit pieces have to do the same, whatever
scales meet inside a row, in any tile that a workgroup takes. Each output may
be off by 2^-21 of the sum of its terms' magnitudes (roundings of at most
4096 terms and what the pieces leave out of each); selections and products of
whole numbers below 2^24 are exact.
"""

from __future__ import annotations

import numpy as np
import pytest

from test_split_products import _call, _check, _conv, _gemm

pytestmark = pytest.mark.gpu

# (m, n, k, nt): 128x128, 128x64 (unaligned) and 64x64 tiles, and short
# products on 32x32 tiles (aligned, unaligned)
PRODUCTS = [(1500, 1100, 640, True), (1500, 1100, 640, False), (1999, 2001, 333, True), (700, 900, 544, False),
            (64, 352, 1120, True), (129, 300, 263, True)]


def _uniform(rng, *shape):
    return rng.uniform(-1, 1, shape).astype(np.float32)


# (a row block at `scale`, K): K within the first 16, one past it, and
# operands that are nonzero only there
@pytest.mark.parametrize("scale", [1e-6, 1e-9, 1e-12])
@pytest.mark.parametrize("k,used", [(5, 5), (16, 16), (17, 17), (64, 16), (160, 16)])
def test_later_tiles_of_a_workgroup(k, used, scale, hip, abi):
    """4096 x 4096 outputs: every workgroup has several tiles, ordinary ones
    first and small ones after."""
    print(f"case gemm 4096x4096x{k} used {used} scale {scale}", flush=True)
    rng = np.random.default_rng(k)
    a, b = _uniform(rng, 4096, k), _uniform(rng, k, 4096)
    a[2048:] *= np.float32(scale)
    a[:, used:] = 0
    _check(_gemm(hip, abi, a, b, True), a, b, f"K {k} scale {scale}")


@pytest.mark.parametrize("scale", [1e-7, 1e-10])
def test_later_pixels_of_a_workgroup(scale, hip, abi):
    """1x1 convolution of 32 channels, the last 16 of them zero in the later
    images' pixels."""
    print(f"case conv 1x1 scale {scale}", flush=True)
    rng = np.random.default_rng(5)
    x = rng.standard_normal((64, 32, 56, 56)).astype(np.float32)
    x[32:] *= np.float32(scale)
    x[32:, 16:] = 0
    w = rng.standard_normal((64, 1, 1, 32)).astype(np.float32)
    _check(*_conv(hip, abi, x, w, 1, 0), f"scale {scale}")


def _mixed(rng, which, m, n, k):
    """Elements of very different size within a row; what the large ones
    meet is zero, so that the small ones make the result."""
    a, b = _uniform(rng, m, k), _uniform(rng, k, n)
    big = np.arange(k) % 4 == 0
    a_small, b_size = {"2^-30": (2.0 ** -30, 3e4), "2^-60": (2.0 ** -60, 3e4), "2^-100": (2.0 ** -100, 2.0 ** 80),
                       "denormal": (2.0 ** -130, 2.0 ** 90), "plain": (2.0 ** -40, 1.0)}[which]
    a[:, ~big] *= np.float32(a_small)
    b[big] = 0
    b[~big] *= np.float32(b_size)
    return a, b


@pytest.mark.parametrize("which", ["2^-30", "2^-60", "2^-100", "denormal", "plain"])
@pytest.mark.parametrize("m,n,k,nt", PRODUCTS)
def test_small_beside_large(m, n, k, nt, which, hip, abi):
    print(f"case gemm {m}x{n}x{k} nt={nt} small beside large {which}", flush=True)
    a, b = _mixed(np.random.default_rng(m + k), which, m, n, k)
    _check(_gemm(hip, abi, a, b, nt), a, b, which)


def _spread(rng, shape, lo, hi):
    """fp32 values with all 24 bits, exponents of [lo, hi]."""
    x = rng.integers(1 << 23, 1 << 24, shape).astype(np.float32) * rng.choice([-1, 1], shape).astype(np.float32)
    return np.ldexp(x, (rng.integers(lo, hi + 1, shape) - 23)).astype(np.float32)


EXPONENTS = {"one": (0, 0), "f16": (-12, 15), "small": (-126, -90), "usual": (-126, 100), "all": (-126, 127)}


@pytest.mark.parametrize("which", sorted(EXPONENTS))
@pytest.mark.parametrize("m,n,k,nt", PRODUCTS)
def test_selection_is_exact(m, n, k, nt, which, hip, abi):
    """Rows of a permutation: the product's rows are the other operand's."""
    print(f"case gemm {m}x{n}x{k} nt={nt} selection of {which}", flush=True)
    rng = np.random.default_rng(m + k)
    pick = rng.integers(0, k, m)
    a = np.zeros((m, k), np.float32)
    a[np.arange(m), pick] = 1
    b = _spread(rng, (k, n), *EXPONENTS[which])
    assert np.array_equal(_gemm(hip, abi, a, b, nt), b[pick])


@pytest.mark.parametrize("m,n,k,nt", PRODUCTS)
def test_whole_numbers_are_exact(m, n, k, nt, hip, abi):
    """One product of two 12-bit numbers per output, sums of some others."""
    print(f"case gemm {m}x{n}x{k} nt={nt} whole numbers", flush=True)
    rng = np.random.default_rng(m)
    a = np.zeros((m, k), np.float32)
    a[np.arange(m), rng.integers(0, k, m)] = rng.integers(2048, 4096, m)
    b = rng.integers(-4095, 4096, (k, n)).astype(np.float32)
    assert np.array_equal(_gemm(hip, abi, a, b, nt), (a.astype(np.float64) @ b).astype(np.float32))
    a = rng.integers(-100, 101, (m, k)).astype(np.float32) * (np.arange(k) < 300)
    b = rng.integers(-500, 501, (k, n)).astype(np.float32)
    assert np.array_equal(_gemm(hip, abi, a, b, nt), (a.astype(np.float64) @ b).astype(np.float32))


# (n, ci, h, w, co, k): tiles of 128x128 and 64x256 (whole, shared); short, in
# pieces (five slices a wave on 392 tiles) and with the fp32 instruction
CONVS = [(16, 256, 28, 27, 128, 1), (32, 64, 56, 56, 64, 3), (8, 256, 14, 14, 256, 3), (2, 64, 56, 56, 64, 3),
         (1, 64, 14, 14, 64, 3), (1, 96, 9, 11, 40, 1)]


@pytest.mark.parametrize("which", sorted(EXPONENTS))
@pytest.mark.parametrize("shape", CONVS, ids=[str(s) for s in CONVS])
def test_selection_by_a_convolution(shape, which, hip, abi):
    n, ci, h, w, co, k = shape
    print(f"case conv {shape} selection of {which}", flush=True)
    rng = np.random.default_rng(ci + h)
    x = _spread(rng, (n, ci, h, w), *EXPONENTS[which])
    pick = rng.integers(0, ci, co)
    v = np.zeros((co, k, k, ci), np.float32)
    v[np.arange(co), k // 2, k // 2, pick] = 1
    got, _, _ = _conv(hip, abi, x, v, 1, k // 2)
    assert np.array_equal(got.reshape(co, n, h, w).transpose(1, 0, 2, 3), x[:, pick])


@pytest.mark.parametrize("which", ["2^-30", "2^-60", "2^-100", "denormal", "plain"])
@pytest.mark.parametrize("shape", CONVS, ids=[str(s) for s in CONVS])
def test_small_beside_large_channels(shape, which, hip, abi):
    n, ci, h, w, co, k = shape
    print(f"case conv {shape} small beside large {which}", flush=True)
    rng = np.random.default_rng(ci + h)
    a, b = _mixed(rng, which, 1, 1, ci)
    x = (_uniform(rng, n, ci, h, w) * np.abs(a.reshape(1, ci, 1, 1))).astype(np.float32)
    v = (_uniform(rng, co, k, k, ci) * np.abs(b.reshape(ci))).astype(np.float32)
    _check(*_conv(hip, abi, x, v, 1, k // 2), f"{shape} {which}")


# (n, ci, h, w, co): with the fp32 instruction, and in pieces (six slices a
# wave on 352 tiles, K % 4 == 3 and 0)
@pytest.mark.parametrize("which", ["2^-30", "plain", "one", "whole", "large", "inf", "nan"])
@pytest.mark.parametrize("shape", [(1, 83, 9, 11, 40), (3, 83, 30, 31, 100), (3, 84, 30, 31, 100)], ids=str)
def test_stored_weights(shape, which, hip, abi):
    """The short kernel of weights as stored."""
    n, ci, h, w, co = shape
    print(f"case stored conv {shape} {which}", flush=True)
    rng = np.random.default_rng(4)
    x, v = _uniform(rng, n, ci, h, w), _uniform(rng, co, ci, 3, 3)
    pick = rng.integers(0, ci, co)
    if which in ("one", "whole"):
        x = _spread(rng, x.shape, 0, 0) if which == "one" else rng.integers(-4095, 4096, x.shape).astype(np.float32)
        v[:] = 0
        v[np.arange(co), pick, 1, 1] = 1 if which == "one" else 4095
    elif which == "large":
        x *= np.float32(1e32)
    elif which == "inf":
        x[0, 5, 4, 6] = np.inf
    elif which == "nan":
        v[7, 80, 0, 2] = np.nan
    else:
        a, b = _mixed(rng, which, 1, 1, ci)
        x *= np.abs(a.reshape(1, ci, 1, 1))
        v *= np.abs(b.reshape(1, ci, 1, 1))
    got = _call(abi, lambda i, u, o, *s: hip.nnc_conv(i, u, None, o, *s), [x, v], (3, 3, 1, 1, 1, 1), (n, co, h, w))
    if which in ("one", "whole"):
        assert np.array_equal(got, x[:, pick] * v[np.arange(co), pick, 1, 1].reshape(1, co, 1, 1))
        return
    xp = np.pad(x, ((0, 0), (0, 0), (1, 1), (1, 1)))
    cols = np.stack([xp[:, :, r:r + h, q:q + w] for r in range(3) for q in range(3)], 2)
    cols = cols.transpose(1, 2, 0, 3, 4).reshape(ci * 9, n * h * w)
    _check(got.transpose(1, 0, 2, 3).reshape(co, -1), v.reshape(co, -1), cols, which)


# ---------------------------------------------------------------------------
# the RGB stem's row kernels (512 output rows of 32 pixels): alone and with
# its max pool
# ---------------------------------------------------------------------------
def _stem_case(which):
    rng = np.random.default_rng(17)
    x = rng.standard_normal((16, 3, 64, 64)).astype(np.float32)
    w = (rng.standard_normal((64, 7, 7, 3)) * np.sqrt(2 / 147)).astype(np.float32)
    if which == "bytes":
        x = rng.integers(0, 256, x.shape).astype(np.float32)
    elif which == "sixteen_bit":
        x = rng.integers(0, 65536, x.shape).astype(np.float32)
    elif which == "huge":
        x *= np.float32(1e32)
    elif which == "tiny":
        x *= np.float32(1e-30)
    elif which == "tiny_rows":
        x[3, :, 20:40] *= np.float32(1e-9)
        x[5] *= np.float32(1e-36)
    elif which == "inf":
        x[2, 1, 30, 30] = np.inf
        x[4, 0, 0, 0] = -np.inf
        x[7, 2, 63, 63] = np.inf
    elif which == "nan":
        x[2, 1, 30, 31] = np.nan
    elif which == "lowest":  # the type's lowest value against zero and small weights
        x[6, 0, 10, 11] = -np.finfo(np.float32).max
        w[:, :, :, 0] *= np.float32(1e-3)
        w[::2, :, :, 0] = 0
    elif which == "tiny_weights":
        w[9] *= np.float32(1e-12)
        w[10] *= np.float32(1e-35)
    elif which == "huge_weights":
        w[9] *= np.float32(1e9)
        w[10] *= np.float32(1e35)
    elif which == "inf_weight":
        w[11, 3, 3, 1] = np.inf
    elif which == "nan_weight":
        w[12, 0, 6, 2] = np.nan
    elif which == "mixed":  # one channel large, its weights zero
        x[:, 1:] *= np.float32(2.0 ** -40)
        w[:, :, :, 0] = 0
    elif which == "mixed_columns":  # the same within pairs of columns
        x[..., 1::2] *= np.float32(2.0 ** -40)
        w[:, :, 1::2] = 0
    elif which == "mixed_weights":
        x[:, 0] *= np.float32(2.0 ** -40)
        w[:, :, :, 1:] *= np.float32(2.0 ** -60)
    elif which in ("select", "select_one"):
        x = _spread(rng, x.shape, *((-126, 60) if which == "select" else (0, 0)))
        w[:] = 0
        w[np.arange(64), rng.integers(0, 7, 64), rng.integers(0, 7, 64), rng.integers(0, 3, 64)] = 1
    return x, w


def _stem_columns(x):
    xp = np.pad(x, ((0, 0), (0, 0), (3, 3), (3, 3)))
    cols = [xp[:, :, r:r + 64:2, q:q + 64:2] for r in range(7) for q in range(7)]  # (tap, channel)
    return np.stack(cols).transpose(0, 2, 1, 3, 4).reshape(147, -1)


STEM = ["unit", "bytes", "sixteen_bit", "huge", "tiny", "tiny_rows", "inf", "nan", "lowest", "tiny_weights",
        "huge_weights", "inf_weight", "nan_weight", "mixed", "mixed_columns", "mixed_weights", "select", "select_one"]


@pytest.mark.parametrize("which", STEM)
def test_stem_rows(which, hip, abi):
    print(f"case stem rows {which}", flush=True)
    x, w = _stem_case(which)
    rows = np.zeros((64, 160), np.float32)
    rows[:, :147] = w.reshape(64, 147)
    got = _call(abi, lambda i, v, o, *s: hip.nnc_hip_conv_packed(i, v, None, None, o, *s), [x, rows],
                (7, 7, 2, 2, 3, 3, 0), (16, 64, 32, 32))
    cols = _stem_columns(x)
    got = got.transpose(1, 0, 2, 3).reshape(64, -1)
    if which.startswith("select"):
        assert np.array_equal(got, (w.reshape(64, 147).astype(np.float64) @ cols).astype(np.float32))
    else:
        _check(got, w.reshape(64, 147), cols, which)
    # the same row with its max pool: the pooled relu of those outputs
    pooled = _call(abi, lambda i, v, o, *s: hip.nnc_hip_conv_maxpool(i, v, None, o, *s), [x, rows], (7, 7, 2, 2, 3, 3),
                   (16, 64, 16, 16))
    relu = np.where(got > 0, got, np.float32(0)).reshape(64, 16, 32, 32).transpose(1, 0, 2, 3)
    rp = np.pad(relu, ((0, 0), (0, 0), (1, 1), (1, 1)))
    want = np.max([rp[:, :, r:r + 32:2, q:q + 32:2] for r in range(3) for q in range(3)], axis=0)
    assert np.array_equal(pooled, want)


# ---------------------------------------------------------------------------
# extents past 32-bit byte offsets
# ---------------------------------------------------------------------------
def test_output_row_of_2_gib(hip, abi):
    m, n = 2, (1 << 29) + 72
    print(f"case gemm_nt {m}x{n}x1", flush=True)
    a = np.array([[3], [-5]], np.float32)
    b = (np.arange(n, dtype=np.int64) % 8191).astype(np.float32).reshape(n, 1)
    got = _call(abi, lambda x, y, o, *s: hip.nnc_gemm_nt(x, y, None, o, *s), [a, b], (1.0, 0.0), (m, n))
    assert np.array_equal(got[0], 3 * b[:, 0]) and np.array_equal(got[1], -5 * b[:, 0])


@pytest.mark.parametrize("k", [1, 3])
def test_output_plane_of_2_gib(k, hip, abi):
    """A plane that reaches far past its image: the bias there."""
    side = 23171
    print(f"case conv {k}x{k} plane {side}", flush=True)
    rng = np.random.default_rng(k)
    x, v = _uniform(rng, 1, 32, 5, 5), _uniform(rng, 1, k, k, 32)
    bias = np.array([0.5], np.float32)
    got = _call(abi, lambda i, w, b, o, *s: hip.nnc_hip_conv_packed(i, w, b, None, o, *s), [x, v, bias],
                (k, k, 1, 1, 0, 0, 0), (1, 1, side, side))[0, 0]
    xp = np.pad(x.astype(np.float64), ((0, 0), (0, 0), (0, k), (0, k)))
    want = sum(np.einsum("c,chw->hw", v[0, r, q].astype(np.float64), xp[0, :, r:r + 5, q:q + 5])
               for r in range(k) for q in range(k)) + 0.5
    assert np.max(np.abs(got[:5, :5] - want)) < 1e-4
    got[:5, :5] = 0.5
    assert np.all(got == np.float32(0.5))
