"""Short convolutions and products on 32 x 32 tiles held in registers
(conv_ws_k, conv_wss_k, gemm_ws_k, gemm_wsu_k): weights as stored, rows off
16-byte boundaries, K that ends inside a 16-byte load, a tile's K split over
workgroups, and operands of any size. The reference is the float64 result; an
output may be off by 2^-21 of the sum of its terms' magnitudes (one rounding
per 2 terms of random signs, K <= 4096).
"""

from __future__ import annotations

import numpy as np
import pytest

from test_split_products import BOUND, _call, _check, _gemm

pytestmark = pytest.mark.gpu


def _scaled(rng, shape, kind):
    x = rng.uniform(-1, 1, shape)
    if kind == "wide":  # rows beyond f16 on both sides, some infinite
        x *= 2.0 ** rng.integers(-40, 40, (shape[0],) + (1,) * (len(shape) - 1))
    return x.astype(np.float32)


@pytest.mark.parametrize("kind", ["unit", "wide"])
@pytest.mark.parametrize("m,n,k,nt", [
    (33, 31, 33, True),       # one slice and one k, every edge
    (2, 65, 131, False),      # unaligned A, x-contiguous B
    (59, 61, 3582, True),     # split over workgroups, K % 4 == 2
    (129, 300, 263, True),    # K % 4 == 3
    (64, 352, 1120, True),    # aligned, split
    (97, 257, 481, False),    # K % 4 == 1
    (400, 700, 45, True),     # unaligned, many tiles: 64 x 64 tiles
])
def test_short_gemm(m, n, k, nt, kind, hip, abi):
    print(f"case short gemm {m}x{n}x{k} nt={nt} {kind}", flush=True)
    rng = np.random.default_rng(m * n + k)
    a, b = _scaled(rng, (m, k), kind), _scaled(rng, (n, k), kind).T
    if kind == "wide":
        a[0, 0] = np.inf
    _check(_gemm(hip, abi, a, np.ascontiguousarray(b), nt), a, b, f"{m}x{n}x{k}")


def _unfold(x, k, s, p):
    n, c, h, w = x.shape
    xp = np.zeros((n, c, h + 2 * p, w + 2 * p))
    xp[:, :, p:p + h, p:p + w] = x
    ho, wo = (h + 2 * p - k) // s + 1, (w + 2 * p - k) // s + 1
    cols = [xp[:, :, r:r + s * ho:s, q:q + s * wo:s] for r in range(k) for q in range(k)]
    return np.stack(cols, 2).reshape(n, c * k * k, ho * wo)


@pytest.mark.parametrize("kind", ["unit", "wide"])
@pytest.mark.parametrize("n,ci,co,h,w,k,s,p", [
    (1, 1, 6, 28, 28, 5, 1, 2),     # one slice
    (1, 6, 16, 14, 14, 5, 1, 0),    # K % 4 == 2, split
    (2, 3, 33, 9, 7, 3, 2, 1),      # K below a slice
    (3, 83, 65, 9, 5, 3, 1, 1),     # K % 4 == 3, split
    (1, 32, 31, 11, 13, 1, 1, 0),   # 1x1, whole slices (tap-major already)
    (2, 35, 40, 8, 9, 1, 2, 0),     # 1x1, strided
    (1, 300, 17, 7, 8, 3, 1, 1),    # long K, many workgroups a tile
    (1, 5, 8, 12, 12, 7, 1, 3),     # 49 taps
    (1, 3, 8, 16, 16, 8, 1, 4),     # 64 taps: the tile kernel
])
def test_stored_conv(n, ci, co, h, w, k, s, p, kind, hip, abi):
    print(f"case stored conv {n}x{ci}->{co} {h}x{w} k{k} s{s} p{p} {kind}", flush=True)
    rng = np.random.default_rng(ci * co + h)
    x, wt = rng.standard_normal((n, ci, h, w)).astype(np.float32), _scaled(rng, (co, ci, k, k), kind)
    bias = rng.standard_normal(co).astype(np.float32)
    cols, rows = _unfold(x.astype(np.float64), k, s, p), wt.reshape(co, -1).astype(np.float64)
    ho, wo = (h + 2 * p - k) // s + 1, (w + 2 * p - k) // s + 1
    want = np.maximum(rows @ cols + bias[:, None], 0).reshape(n, co, ho, wo)
    size = (np.abs(rows) @ np.abs(cols) + np.abs(bias)[:, None]).reshape(n, co, ho, wo)
    got = _call(abi, hip.nnc_conv_relu, [x, wt, bias], (k, k, s, s, p, p), (n, co, ho, wo))
    off = np.abs(got.astype(np.float64) - want) / size
    assert off.max() <= BOUND, f"worst {off.max():.3g}"
