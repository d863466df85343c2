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

import ctypes

import numpy as np
import pytest

from oracle import reference as ref
from test_gpu_kernels import _run_depth, needs_specialised, rng_uniform, run_conv, run_matmul, run_matmul_layout
from xtc_amd.runtimes.hip import capi
from xtc_amd.runtimes.hip.buffer import DeviceBuffer, ensure_device

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


# default calls whose class is a 64x64 or 128x128 tile of four waves and which
# run on an 8-wave one: cut by M, N and K, K split less often than the class says
@pytest.mark.parametrize("trans_b,M,N,K,cls,tile,splits", [
    (False, 1000, 1104, 1200, 64, (128, 128, 32, 2, 4), 3),
    (True, 257, 2308, 2052, 64, (128, 128, 32, 2, 4), 4),
    (True, 258, 4100, 4100, 64, (128, 256, 32, 2, 4), 4),
    (False, 300, 2052, 8196, 64, (128, 128, 32, 2, 4), 5),
    (True, 1284, 4612, 260, 64, (256, 128, 32, 4, 2), 1),
    (False, 2049, 2052, 100, 128, (256, 128, 32, 4, 2), 1),
    (True, 2050, 2308, 1156, 128, (256, 128, 32, 4, 2), 1),
])
def test_default_calls_on_eight_wave_tiles(trans_b, M, N, K, cls, tile, splits):
    print(f"[planes wide] {M}x{N}x{K} trans_b {trans_b}", flush=True)
    d = capi.MatmulDesc(dtype=capi.XTC_HIP_F32, M=M, N=N, K=K, trans_b=int(trans_b))
    assert capi.default_tile("float32", False, M, N, K)[0][0] == cls
    assert capi.matmul_default_tile(d) == (tile, splits)
    a, b = rng_uniform(M + K, (M, K)), rng_uniform(N + K, (K, N))
    out = run_matmul_layout(a, b, "float32", False, trans_b)
    check(out, a, b)
    # the tile and split by name: the same call
    np.testing.assert_array_equal(run_matmul_layout(a, b, "float32", False, trans_b, tile=tile, split_k=splits), out)


# no whole vectors anywhere: fp32 and bf16 rows at element alignment, units cut
# by K and N, tiles cut by M and N, split-K partial rows of whole vectors
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("M,N,K,split", [(1, 1, 33, 1), (3, 5, 37, 1), (64, 65, 63, 1), (67, 129, 131, 1),
                                         (130, 63, 257, 2), (65, 71, 515, 0), (33, 1021, 777, 0)])
def test_any_alignment(dtype, M, N, K, split):
    print(f"[planes any] {dtype} {M}x{N}x{K} split {split}", flush=True)
    a, b = rng_uniform(M + K, (M, K)), rng_uniform(N + K, (K, N))
    if dtype == "bfloat16":
        a, b = ref.round_bf16(a), ref.round_bf16(b)
    bias = rng_uniform(7, (N,))
    out = run_matmul(a, b, dtype, split_k=split, relu=True, thr=-1.0, bias=bias)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    want = np.maximum(a64 @ b64 + bias, -1.0)
    # bf16 products are exact: at most one rounding per product and per split
    terms = K / 32 + 17 if dtype == "float32" else K + 17
    assert np.all(np.abs(out - want) <= terms * 2.0**-24 * (np.abs(a64) @ np.abs(b64) + 1))
    ai, bi = ref.np_init((M, K), "float32"), ref.np_init((K, N), "float32")
    np.testing.assert_array_equal(run_matmul(ai, bi, dtype, split_k=split), ai.astype(np.float64) @ bi)


def test_splitwave_behind_64x64x32():
    # the same splits in the same order as the template, which runs 80 rows (no
    # whole 32-row blocks): its rows bit for bit, at both depths
    a, b = rng_uniform(3, (96, 512)), rng_uniform(4, (512, 160))
    template = _run_depth(a[:80].copy(), b, "float32", (64, 64, 32, 2, 2), 4, 0, False)
    for depth in (0, 2, 4):
        np.testing.assert_array_equal(_run_depth(a, b, "float32", (64, 64, 32, 2, 2), 4, depth, False)[:80], template)


# B stored transposed, read in place: rows of B^T cut by N, slabs cut by K
@pytest.mark.parametrize("dtype,tile", [("float32", TILES[0]), ("float32", TILES[1]), ("float32", TILES[2]),
                                        ("float32", (64, 64, 32, 2, 2)), ("bfloat16", (64, 64, 64, 2, 2)),
                                        ("bfloat16", (128, 128, 64, 2, 2))])
@pytest.mark.parametrize("M,N,K,split", [(1, 8, 8, 1), (130, 264, 136, 1), (257, 136, 1048, 3)])
def test_transposed_b(dtype, tile, M, N, K, split):
    print(f"[planes bt] {dtype} {tile} {M}x{N}x{K} split {split}", flush=True)
    ai, bi = ref.np_init((M, K), "float32"), ref.np_init((K, N), "float32")[::-1].copy()
    for bt in (True, False):
        out = run_matmul_layout(ai, bi, dtype, False, bt, tile=tile, split_k=split, pad_a=8, pad_b=16)
        np.testing.assert_array_equal(out, ai.astype(np.float64) @ bi)


# B^T in place with bias and relu in the epilogue and in the finishing workgroup
@pytest.mark.parametrize("dtype,tile", [("float32", TILES[2]), ("float32", (64, 64, 32, 2, 2)),
                                        ("bfloat16", (64, 64, 64, 2, 2)), ("bfloat16", (128, 128, 64, 2, 2))])
@pytest.mark.parametrize("split", [1, 2])
def test_transposed_b_bias_relu(dtype, tile, split):
    M, N, K = 130, 264, 1048
    ai, bi = ref.np_init((M, K), "float32"), ref.np_init((K, N), "float32")[::-1].copy() - 4
    bias = (np.arange(N) % 9 - 4).astype(np.float32)
    out = run_matmul_layout(ai, bi, dtype, False, True, tile=tile, split_k=split, relu=True, bias=bias)
    np.testing.assert_array_equal(out, np.maximum(ai.astype(np.float64) @ bi + bias, 0))


# bf16 workgroups of 4 or 8 waves (512 and 520 of them); 128-row tiles whose
# splits pass the 256 CUs (462 and 264 workgroups), fit them with fewer than 8
# slabs, and fit them on two k-groups (198 workgroups of 12, 12 and 10 slabs, the
# last one cut by K; 256 of 11 slabs, 6 and 5 a group)
@pytest.mark.parametrize("tile,M,N,K,split", [((64, 64, 64, 2, 2), 1024, 2048, 136, 1), ((64, 64, 64, 2, 2), 505, 4136, 136, 1),
                                              ((64, 64, 64, 2, 2), 505, 2088, 264, 2), ((128, 128, 64, 2, 2), 129, 4104, 1160, 8),
                                              ((128, 128, 64, 2, 2), 256, 4224, 256, 4),
                                              ((128, 128, 64, 2, 2), 256, 4224, 1160, 3),
                                              ((128, 128, 64, 2, 2), 256, 4224, 2120, 3),
                                              ((128, 128, 64, 2, 2), 250, 4088, 2816, 4)])
def test_bf16_workgroups_and_splits(tile, M, N, K, split):
    print(f"[planes bf16] {tile} {M}x{N}x{K} split {split}", flush=True)
    ai, bi = ref.np_init((M, K), "float32"), ref.np_init((K, N), "float32")[::-1].copy()
    for bt in (True, False):
        out = run_matmul_layout(ai, bi, "bfloat16", False, bt, tile=tile, split_k=split)
        np.testing.assert_array_equal(out, ai.astype(np.float64) @ bi)


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


@pytest.mark.parametrize("exp", [-126, -120, -117])
@pytest.mark.parametrize("tile", [TILES[0], (64, 64, 32, 2, 2)])
def test_small_normal_operands_that_cancel(tile, exp):
    # normal operands below 2^-110 lose the bits below 2^-133: x and 2^exp
    # have the same planes, so that every sum of the planes is exactly zero,
    # where the product with 2^100 is not
    M, N, K = (8, 8, 96) if tile[0] == 256 else (1500, 1500, 256)
    a, b = np.zeros((M, K), np.float32), np.full((K, N), 2.0**100, np.float32)
    x = np.ldexp(1 + 2.0 ** -np.arange(exp + 135, 24), exp).astype(np.float32)
    for i in range(M):
        k = (7 * i) % (K - 1)
        a[i, k], a[i, k + 1] = x[i % len(x)], -np.float32(2.0**exp)
    b[:, 1::2] = 2.0**-3
    check(run_matmul(a, b, tile=tile, split_k=1), a, b)


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


def test_small_tile_edges():
    # 64x64x32 runs here from 512 workgroups of 8 slabs unsplit, and of 4 slabs
    # from 1152 with K split
    for M, N, K in ((1400, 1540, 260), (2050, 1028, 1000)):
        a, b = rng_uniform(M, (M, K)), rng_uniform(N, (K, N))
        check(run_matmul(a, b, tile=(64, 64, 32, 2, 2), split_k=1), a, b)
    a, b = rng_uniform(8, (1004, 1200)), rng_uniform(9, (1200, 1104))
    check(run_matmul(a, b, tile=(64, 64, 32, 2, 2), split_k=8), a, b)


def check_conv(dtype, n, h, w, c, f, r, s, stride, pads, pad_value, tile, split):
    print(f"[planes conv] {dtype} {(n, h, w, c, f, r, s)} stride {stride} pads {pads} {tile} split {split}", flush=True)
    rng = np.random.default_rng(h * w + c)
    x = rng.integers(-3, 4, (n, h, w, c)).astype(np.float32)
    wt = rng.integers(-2, 3, (r, s, c, f)).astype(np.float32)
    bias = rng.integers(-2, 3, f).astype(np.float32)
    out = run_conv(x, wt, dtype, stride, pads, pad_value, tile, split_k=split, bias=bias)
    xp = ref.pad(x, [(0, 0), pads[:2], pads[2:], (0, 0)], pad_value)
    np.testing.assert_array_equal(out, (ref.conv2d(xp, wt, stride) + bias).astype(np.float32))


# channels and filters of no whole vector: windows that leave the image on
# every side, runs of S C elements shorter and longer than a unit and a slab
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("n,h,w,c,f,r,s,stride,pads,pad_value,split", [
    (1, 5, 4, 35, 1, 1, 1, (1, 1), (0, 0, 0, 0), 0.0, 0),
    (2, 9, 7, 3, 64, 3, 3, (1, 1), (1, 1, 1, 1), 0.0, 1),
    (1, 17, 15, 3, 24, 7, 7, (2, 2), (3, 2, 1, 3), 2.0, 2),
    (1, 12, 11, 5, 7, 2, 3, (2, 1), (1, 0, 2, 1), -1.0, 0),
    (1, 10, 10, 37, 66, 3, 3, (1, 2), (0, 2, 1, 0), 0.0, 3),
    (3, 70, 72, 3, 72, 3, 3, (1, 1), (1, 1, 1, 1), 1.0, 1),
])
def test_conv_any_alignment(dtype, n, h, w, c, f, r, s, stride, pads, pad_value, split):
    check_conv(dtype, n, h, w, c, f, r, s, stride, pads, pad_value, None, split)
    for tile in ((64, 64, 32, 2, 2), (128, 64, 32, 4, 2)) if dtype == "float32" else ((64, 64, 64, 2, 2),):
        check_conv(dtype, n, h, w, c, f, r, s, stride, pads, pad_value, tile, split)


@pytest.mark.parametrize("dtype,tile", [("bfloat16", (64, 64, 64, 2, 2)), ("bfloat16", (128, 64, 64, 2, 2)),
                                        ("bfloat16", (128, 128, 64, 2, 2)), ("float32", (64, 64, 32, 2, 2)),
                                        ("float32", (64, 64, 16, 2, 2))])
@pytest.mark.parametrize("n,h,w,c,f,r,s,stride,pads,pad_value,split", [
    (1, 9, 10, 8, 8, 1, 1, (1, 1), (0, 0, 0, 0), 0.0, 1),
    (2, 13, 11, 24, 72, 3, 3, (2, 1), (1, 2, 0, 1), 2.0, 2),
    (1, 182, 182, 32, 40, 3, 3, (1, 1), (1, 1, 1, 1), -1.0, 1),
])
def test_conv_vectors(dtype, tile, n, h, w, c, f, r, s, stride, pads, pad_value, split):
    check_conv(dtype, n, h, w, c, f, r, s, stride, pads, pad_value, tile, split)


def test_conv_infinite_pad():
    x, wt = np.ones((1, 6, 6, 3), np.float32), np.ones((3, 3, 3, 8), np.float32)
    out = run_conv(x, wt, "float32", (1, 1), (1, 1, 1, 1), float("inf"))
    want = np.full((1, 6, 6, 8), np.inf, np.float32)
    want[:, 1:5, 1:5] = 27
    np.testing.assert_array_equal(out, want)


def test_captured_ragged_calls_keep_no_growable_scratch():
    # an eager call splits K and leaves the stream's workspace behind, the
    # captured one runs unsplit; a larger call then replaces the workspace
    # between replays
    L = capi.lib()
    # the HIP runtime this process runs on
    hip = ctypes.CDLL(next(ln.split()[-1] for ln in open("/proc/self/maps") if "libamdhip64" in ln))
    stream = ctypes.c_void_p(L.xtc_hip_stream_create())
    M, N, K = 130, 253, 515
    a, b = rng_uniform(21, (M, K)), rng_uniform(22, (K, N))
    A, B = DeviceBuffer.from_numpy(a), DeviceBuffer.from_numpy(b)
    C, E = DeviceBuffer(M * N * 4), DeviceBuffer(M * N * 4)
    big = DeviceBuffer(1021 * 1021 * 4)
    big.zero()

    def call(out, m, n, k, x, y, split):
        d = capi.MatmulDesc(dtype=capi.XTC_HIP_F32, M=m, N=n, K=k, split_k=split, stream=stream, xcd_remap=1)
        d.tile = capi.Tile(64, 64, 32, 2, 2)
        capi.check(L.xtc_hip_matmul(ctypes.byref(d), x.c_ptr, y.c_ptr, out.c_ptr, None), "matmul")

    def ok(code):
        assert code == 0, code

    def eager(split):
        call(E, M, N, K, A, B, split)
        capi.check(L.xtc_hip_stream_synchronize(stream), "sync")
        return E.to_numpy((M, N), np.float32)

    split4, unsplit = eager(4), eager(1)
    check(split4, a, b)
    graph, run = ctypes.c_void_p(), ctypes.c_void_p()
    ok(hip.hipStreamBeginCapture(stream, 1))
    call(C, M, N, K, A, B, 4)
    ok(hip.hipStreamEndCapture(stream, ctypes.byref(graph)))
    ok(hip.hipGraphInstantiate(ctypes.byref(run), graph, None, None, ctypes.c_size_t(0)))
    for _ in range(4):
        C.zero()
        capi.check(L.xtc_hip_synchronize(), "sync")
        ok(hip.hipGraphLaunch(run, stream))
        capi.check(L.xtc_hip_stream_synchronize(stream), "sync")
        np.testing.assert_array_equal(C.to_numpy((M, N), np.float32), unsplit)
        out = DeviceBuffer(1021 * 1021 * 4)
        call(out, 1021, 1021, 1021, big, big, 8)
        np.testing.assert_array_equal(eager(4), split4)
    ok(hip.hipGraphExecDestroy(run))
    ok(hip.hipGraphDestroy(graph))
    capi.check(L.xtc_hip_stream_destroy(stream), "destroy")
