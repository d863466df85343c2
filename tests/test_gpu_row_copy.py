# SPDX-License-Identifier: BSD-3-Clause
"""row_copy_kernel (pad and unpad of four elements per thread) where its groups
of four are cut: rows shorter than a group, pads and crops that start and end
inside one, empty interiors, every rank; bit-exact against the oracle."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from oracle import reference as ref
from xtc_amd.runtimes.hip import capi
from xtc_amd.runtimes.hip.buffer import DeviceBuffer, ensure_device

pytestmark = pytest.mark.gpu

CASES = [
    ((1,), [(0, 2)]),
    ((3,), [(1, 0)]),
    ((5, 7), [(1, 2), (3, 1)]),
    ((4, 1), [(0, 0), (2, 3)]),
    ((2, 3, 8), [(0, 1), (2, 0), (4, 4)]),
    ((3, 1, 2, 9), [(1, 1), (0, 3), (1, 0), (5, 2)]),
    ((1, 2, 1, 3, 2, 1, 2, 6), [(0, 1), (1, 0), (0, 0), (1, 1), (0, 2), (1, 0), (0, 0), (1, 3)]),
    ((129, 1030), [(2, 2), (1, 3)]),
]


@pytest.fixture(scope="module", autouse=True)
def device():
    ensure_device(0)
    yield


def _i64(values):
    return (ctypes.c_int64 * len(values))(*values)


@pytest.mark.parametrize("shape,pads", CASES)
def test_pad_and_crop_back(shape, pads):
    rng = np.random.default_rng(len(shape))
    nd, before, after = len(shape), [p[0] for p in pads], [p[1] for p in pads]
    L = capi.lib()
    for dt, call, value in ((np.float32, L.xtc_hip_pad, ctypes.c_float(-2.5)),
                            (np.float64, L.xtc_hip_pad_f64, ctypes.c_double(-2.5))):
        x = rng.uniform(-1, 1, shape).astype(dt)
        want = ref.pad(x, pads, -2.5)
        X, Y, Z = DeviceBuffer.from_numpy(x), DeviceBuffer(want.nbytes), DeviceBuffer(x.nbytes)
        capi.check(call(X.c_ptr, Y.c_ptr, nd, _i64(shape), _i64(before), _i64(after), value, None))
        capi.check(L.xtc_hip_unpad(Y.c_ptr, Z.c_ptr, x.itemsize, nd, _i64(want.shape), _i64(before), _i64(after), None))
        capi.check(L.xtc_hip_synchronize())
        np.testing.assert_array_equal(Y.to_numpy(want.shape, dt), want)
        np.testing.assert_array_equal(Z.to_numpy(shape, dt), x)


@pytest.mark.parametrize("shape,pads", [c for c in CASES if c[0][-1] > 1])
def test_crop_of_16_bit_words(shape, pads):
    x = np.random.default_rng(3).integers(0, 2**16, [s + a + b for s, (a, b) in zip(shape, pads)]).astype(np.uint16)
    want = ref.unpad(x, pads)
    X, Y = DeviceBuffer.from_numpy(x), DeviceBuffer(want.nbytes)
    capi.check(capi.lib().xtc_hip_unpad(X.c_ptr, Y.c_ptr, 2, len(shape), _i64(x.shape), _i64([p[0] for p in pads]),
                                        _i64([p[1] for p in pads]), None))
    capi.check(capi.lib().xtc_hip_synchronize())
    np.testing.assert_array_equal(Y.to_numpy(want.shape, np.uint16), want)
