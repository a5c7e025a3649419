"""Convolutions and products on the 16-bit matrix units (csrc/split_tile.h).

Sizes at the edges of tiles, 16-k steps and 32-k slices, and values outside
the range of the pieces, where a workgroup computes its segment again with
the fp32 instruction. The reference is the float64 product; each output may
be off by 2^-21 of the sum of its terms' magnitudes: 2^-24 of each term that
the pieces leave out, one fp32 rounding per 16 terms (per 2 with the fp32
instruction), K <= 4096, on random signs.
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BOUND = 2.0 ** -21


def _call(abi, fn, arrays, scalars, out_shape):
    from nnc_py_amd import runtime
    bufs = [None if a is None else runtime.DeviceBuffer.from_array(np.ascontiguousarray(a)) for a in arrays]
    out = runtime.DeviceBuffer.empty(out_shape)
    ts = [None if b is None else b.tensor() for b in bufs] + [out.tensor()]
    fn(*[None if t is None else ctypes.byref(t[0]) for t in ts], *scalars)
    runtime.sync()
    code, msg = runtime.last_error()
    assert code == 0, msg
    got = out.to_array()
    for b in bufs + [out]:
        if b is not None:
            b.free()
    return got


def _check(got, a, b, what):
    """got against a @ b in float64; infinities and NaN where fp32 products give them."""
    with np.errstate(all="ignore"):
        a64, b64 = a.astype(np.float64), b.astype(np.float64)
        want, size = a64 @ b64, np.abs(a64) @ np.abs(b64)
    fin = np.isfinite(size)
    assert np.array_equal(np.isnan(got), np.isnan(want)), f"{what}: NaN elsewhere"
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)].astype(np.float32)), f"{what}: infinities differ"
    off = np.abs(got[fin].astype(np.float64) - want[fin])
    bad = off > BOUND * size[fin] + 1e-37
    assert not bad.any(), f"{what}: {bad.sum()} outputs off, worst {np.max(off / np.maximum(size[fin], 1e-300)):.3g}"


def _gemm(hip, abi, a, b, nt):
    m, n = a.shape[0], b.shape[1]
    if nt:
        return _call(abi, lambda x, y, o, *s: hip.nnc_gemm_nt(x, y, None, o, *s), [a, b.T], (1.0, 0.0), (m, n))
    return _call(abi, lambda x, y, o, *s: hip.nnc_gemm(x, y, None, o, *s), [a, b], (1.0, 0.0, 0, 0), (m, n))


GEMM_EDGES = [
    (2048, 1024, 256),   # whole 64x64 tiles
    (1500, 1100, 640),   # shared tiles, ragged rows and columns
    (2049, 1025, 272),   # K ends in the first half of a slice, unaligned N
    (4000, 300, 2000),   # the same with shared 128x128 tiles
    (1999, 2001, 333),   # no alignment anywhere, 128x64 tiles
    (1001, 999, 321),    # K one past a slice
    (2048, 2048, 544),   # whole 128x128 tiles, 17 slices
    (513, 520, 4000),    # many partials per tile
]


@pytest.mark.parametrize("m,n,k", GEMM_EDGES)
@pytest.mark.parametrize("nt", [False, True])
def test_gemm_edges(m, n, k, nt, hip, abi):
    print(f"case gemm {m}x{n}x{k} nt={nt}", flush=True)
    rng = np.random.default_rng(m + k)
    a, b = rng.uniform(-1, 1, (m, k)).astype(np.float32), rng.uniform(-1, 1, (k, n)).astype(np.float32)
    _check(_gemm(hip, abi, a, b, nt), a, b, f"{m}x{n}x{k}")


# (m, n, k, transposed A, transposed B): K a multiple of 4 and no more (both
# loaders of either operand), K past 16 by 4; one round of fp32 tiles on one
# workgroup per CU, shared and whole; unaligned rows over two slices on just
# more than four rounds of 64x64 tiles
GEMM_ROUTES = [(1500, 1100, 644, ta, tb) for ta in (0, 1) for tb in (0, 1)] + [
    (700, 900, 564, 0, 1), (495, 320, 3072, 0, 0), (355, 2592, 1152, 0, 1), (1862, 2348, 41, 0, 0)]


@pytest.mark.parametrize("m,n,k,ta,tb", GEMM_ROUTES)
def test_gemm_routes(m, n, k, ta, tb, hip, abi):
    print(f"case gemm {m}x{n}x{k} ta={ta} tb={tb}", flush=True)
    rng = np.random.default_rng(m + k)
    a, b = rng.uniform(-1, 1, (m, k)).astype(np.float32), rng.uniform(-1, 1, (k, n)).astype(np.float32)
    c = rng.uniform(-1, 1, n).astype(np.float32)
    got = _call(abi, lambda x, y, z, o, *s: hip.nnc_gemm(x, y, z, o, *s), [a.T if ta else a, b.T if tb else b, c],
                (1.0, 1.0, ta, tb), (m, n))
    _check(got, np.hstack([a, np.ones((m, 1), np.float32)]), np.vstack([b, c]), f"{m}x{n}x{k}")


def _scaled(which, a, b):
    if which == "small":
        a *= 1e-6
    elif which == "large":
        a *= 1e7
        b *= 3e5
    elif which == "small_row":
        a[3] *= 1e-7
    elif which == "large_row":
        a[700] *= 1e12
    elif which == "small_column":
        b[:, 500] *= 1e-9
    elif which == "extremes":
        a *= 1e-18
        b *= 1e18
    elif which == "zero_rows":
        a[5:9] = 0
        b[:, 17] = 0
    elif which == "inf":
        a[5, 7] = np.inf
        b[9, 40] = -np.inf
        a[6, 9] = 0  # 0 * -inf
    elif which == "nan":
        a[5, 7] = np.nan
    elif which == "flt_max":  # a mask value against zeros and ordinary numbers
        a[400, 300] = -np.finfo(np.float32).max
        b[300, ::2] = 0
        b[300, 1::2] = 1e-3
    elif which == "in_last_slice":
        a[:, -1] = 1e6
    return a, b


RANGES = ["small", "large", "small_row", "large_row", "small_column", "extremes", "zero_rows", "inf", "nan", "flt_max",
          "in_last_slice"]


@pytest.mark.parametrize("which", RANGES)
@pytest.mark.parametrize("m,n,k", [(1500, 1100, 640), (1999, 2001, 333)])
def test_gemm_ranges(which, m, n, k, hip, abi):
    print(f"case gemm range {which} {m}x{n}x{k}", flush=True)
    rng = np.random.default_rng(7)
    a, b = _scaled(which, rng.uniform(-1, 1, (m, k)).astype(np.float32), rng.uniform(-1, 1, (k, n)).astype(np.float32))
    _check(_gemm(hip, abi, a, b, True), a, b, which)


def _unfold(x, k, stride, pad):
    """im2col, k = (tap, channel): [kh*kw*C, N*Ho*Wo]."""
    n, c, h, w = x.shape
    ho, wo = (h + 2 * pad - k) // stride + 1, (w + 2 * pad - k) // stride + 1
    xp = np.zeros((n, c, h + 2 * pad, w + 2 * pad), x.dtype)
    xp[:, :, pad:pad + h, pad:pad + w] = x
    cols = [xp[:, :, r:r + stride * ho:stride, q:q + stride * wo:stride] for r in range(k) for q in range(k)]
    return np.stack(cols).transpose(0, 2, 1, 3, 4).reshape(k * k * c, n * ho * wo), ho, wo


def _conv(hip, abi, x, w, stride, pad):
    """w [Co][k][k][Ci]; output as [Co, N*Ho*Wo]."""
    co, k = w.shape[0], w.shape[1]
    cols, ho, wo = _unfold(x, k, stride, pad)
    got = _call(abi, lambda i, v, o, *s: hip.nnc_hip_conv_packed(i, v, None, None, o, *s), [x, w],
                (k, k, stride, stride, pad, pad, 0), (x.shape[0], co, ho, wo))
    return got.transpose(1, 0, 2, 3).reshape(co, -1), w.reshape(co, -1), cols


CONV_EDGES = [
    (5, 64, 57, 57, 64, 3, 1),    # Co 64, odd planes: 64x64 tiles
    (32, 64, 56, 56, 64, 3, 1),   # 64x256 tiles, whole
    (32, 32, 41, 43, 40, 3, 1),   # 64x256 tiles past Co and past the pixels
    (9, 96, 29, 31, 130, 3, 2),   # one row past a 128 tile, stride 2
    (8, 256, 14, 14, 256, 3, 1),  # shared tiles
    (16, 256, 28, 27, 128, 1, 1),  # 1x1, whole 128x128 tiles
]


@pytest.mark.parametrize("shape", CONV_EDGES, ids=[str(s) for s in CONV_EDGES])
def test_conv_edges(shape, hip, abi):
    n, ci, h, w, co, k, stride = shape
    print(f"case conv {shape}", flush=True)
    rng = np.random.default_rng(ci + h)
    x = rng.standard_normal((n, ci, h, w)).astype(np.float32)
    v = (rng.standard_normal((co, k, k, ci)) * np.sqrt(2 / (ci * k * k))).astype(np.float32)
    _check(*_conv(hip, abi, x, v, stride, k // 2), str(shape))


@pytest.mark.parametrize("which", ["small", "large", "image", "channel", "inf", "nan", "sparse"])
def test_conv_ranges(which, hip, abi):
    print(f"case conv range {which}", flush=True)
    rng = np.random.default_rng(3)
    x = rng.standard_normal((8, 128, 28, 28)).astype(np.float32)
    v = (rng.standard_normal((128, 3, 3, 128)) * 0.04).astype(np.float32)
    if which == "small":
        x *= 1e-8
    elif which == "large":
        x *= 1e9
    elif which == "image":
        x[3] *= 1e-6
    elif which == "channel":
        v[17] *= 1e-6
    elif which == "inf":
        x[2, 5, 9, 9] = np.inf
    elif which == "nan":
        v[5, 1, 1, 7] = np.nan
    elif which == "sparse":  # pixels whose only nonzero is small
        x[:] = 0
        x[:, 64, ::3, ::3] = 1e-5
        x[0] = 1
    _check(*_conv(hip, abi, x, v, 1, 1), which)


def test_outputs_of_2_gib(hip, abi):
    """Row, image and channel ranges of outputs past 32-bit byte offsets."""
    from nnc_py_amd import runtime
    rng = np.random.default_rng(9)
    print("case gemm 2 GiB", flush=True)
    m, n, k = 33000, 16400, 32
    a, b = rng.uniform(-1, 1, (m, k)).astype(np.float32), rng.uniform(-1, 1, (n, k)).astype(np.float32)
    got = _call(abi, lambda x, y, o, *s: hip.nnc_gemm_nt(x, y, None, o, *s), [a, b], (1.0, 0.0), (m, n))
    rows = [0, 1, 32734, 32735, 32736, m - 1]
    _check(got[rows], a[rows], b.T, "gemm rows")
    del got
    for images, co in ((3, 512), (1, 1500)):
        print(f"case conv 2 GiB, {images} images", flush=True)
        x = rng.standard_normal((images, 32, 600, 601)).astype(np.float32)
        v = rng.standard_normal((co, 1, 1, 32)).astype(np.float32)
        res = _call(abi, lambda i, w, o, *s: hip.nnc_hip_conv_packed(i, w, None, None, o, *s), [x, v],
                    (1, 1, 1, 1, 0, 0, 0), (images, co, 600, 601))
        for i in range(images):
            for c in (0, co // 2, co - 1):
                _check(res[i, c:c + 1].reshape(1, -1), v[c].reshape(1, 32), x[i].reshape(32, -1), f"image {i} channel {c}")
        del res
    assert runtime.last_error()[0] == 0
