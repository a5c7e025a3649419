"""Products and convolutions over the whole range of fp32 values.

Whatever a kernel does about operands outside a range, it has to do in every
tile that a workgroup takes. Each output may be off by 2^-21 of the sum of its
terms' magnitudes (roundings of at most 4096 terms and what 16-bit pieces
leave out of each).
"""

from __future__ import annotations

import numpy as np
import pytest

from test_split_products import _check, _conv, _gemm

pytestmark = pytest.mark.gpu


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
