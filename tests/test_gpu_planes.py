# SPDX-License-Identifier: BSD-3-Clause
"""gemm_planes (xtc_amd/csrc/gemm_planes.hpp): fp32 products on bf16 matrix
instructions, at the edges of its tiles and slabs and over the values its
three bf16 planes cannot hold.

Bound against float64, element by element, with S = sum_k |a| |b|:
  (K / 32 + 16) 2^-24 S + K 2^-148
one fp32 rounding per 32 products and at most one per split (<= 8), the six
products of a slab rounded within its own sum and the dropped ones at 2^-24
of a product each; 2^-148 for sums in the denormal range.
"""

from __future__ import annotations

import numpy as np
import pytest

from test_gpu_kernels import needs_specialised, rng_uniform, run_matmul
from xtc_amd.runtimes.hip.buffer import ensure_device

pytestmark = [pytest.mark.gpu, needs_specialised]

TILES = [(256, 128, 32, 4, 2), (128, 256, 32, 2, 4), (128, 128, 32, 2, 4)]


@pytest.fixture(scope="module", autouse=True)
def device():
    ensure_device(0)
    yield


def check(out, a, b):
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    want = a64 @ b64
    K = a.shape[1]
    bound = (K / 32 + 16) * 2.0**-24 * (np.abs(a64) @ np.abs(b64)) + K * 2.0**-148
    over = np.abs(out - want) - bound
    assert np.all(over <= 0), (np.unravel_index(np.argmax(over), over.shape), np.max(over))


# one and two slabs, the first K with a full pipeline step (96), a slab cut by
# K, splits of unequal depth; one row and one vector, tiles cut in M and in N
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M,N,K,split", [(1, 4, 4, 1), (256, 256, 32, 1), (257, 260, 64, 1), (255, 132, 96, 1),
                                         (300, 516, 100, 1), (129, 388, 1156, 3), (512, 256, 1024, 2)])
def test_edges(tile, M, N, K, split):
    print(f"[planes] {tile} {M}x{N}x{K} split {split}", flush=True)
    a, b = rng_uniform(M + K, (M, K)), rng_uniform(N + K, (K, N))
    check(run_matmul(a, b, tile=tile, split_k=split), a, b)


def test_half_zero_and_wide_operands():
    # relu'd activations, and magnitudes spread over 2^-40 .. 2^40 in one sum
    rng = np.random.default_rng(5)
    a = np.maximum(rng.normal(0, 1, (130, 512)), 0).astype(np.float32)
    b = (rng.normal(0, 1, (512, 256)) * 2.0 ** rng.integers(-40, 41, (512, 1))).astype(np.float32)
    check(run_matmul(a, b, tile=TILES[2], split_k=1), a, b)


@pytest.mark.parametrize("scale_a,scale_b", [(1e-20, 1e-20), (1e-38, 1.0), (1e-42, 1e3), (3e38, 1e-3), (1e30, 1e-35)])
def test_operands_near_the_ends_of_the_range(scale_a, scale_b):
    # uniform in [-1, 1) times the scale: denormals, values whose lower planes
    # fall below bf16's range, values next to the largest
    a = rng_uniform(1, (128, 96)) * np.float32(scale_a)
    b = rng_uniform(2, (96, 128)) * np.float32(scale_b)
    check(run_matmul(a, b, tile=TILES[2], split_k=1), a, b)


def test_infinities_and_nan():
    rng = np.random.default_rng(9)
    a = rng.integers(1, 5, (256, 160)).astype(np.float32)
    b = rng.integers(1, 5, (160, 128)).astype(np.float32)
    a[3, 7], a[200, 100], a[77, 159] = np.inf, -np.inf, np.nan
    a[90, 5], a[90, 6] = np.inf, -np.inf
    a[40, 0] = np.finfo(np.float32).max
    b[7, 9], b[31, 64] = 0.0, -np.finfo(np.float32).max
    with np.errstate(all="ignore"):
        want = (a.astype(np.float64) @ b.astype(np.float64)).astype(np.float32)
    for tile in TILES:
        out = run_matmul(a, b, tile=tile, split_k=1)
        np.testing.assert_array_equal(np.isnan(out), np.isnan(want))
        np.testing.assert_array_equal(np.isposinf(out), np.isposinf(want))
        np.testing.assert_array_equal(np.isneginf(out), np.isneginf(want))
        fin = np.isfinite(want)
        np.testing.assert_allclose(out[fin], want[fin], rtol=160 * 2.0**-24)
