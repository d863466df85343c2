# SPDX-License-Identifier: BSD-3-Clause
"""Which kernels a call of the C-ABI launches, with how many splits of K, and
what scratch it takes, on the CPU: libxtc_hip.so runs against a stand-in for the
HIP runtime (tests/hip_stub/fake_hip.cpp) that records launches and can refuse
memory or report a stream as being captured."""

from __future__ import annotations

import json
import shutil
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
LIB = ROOT / "xtc_amd" / "lib" / "libxtc_hip.so"

pytestmark = pytest.mark.skipif(shutil.which("g++") is None or not LIB.exists(), reason="needs g++ and libxtc_hip.so")

# defines for the scripts: matmul()/conv() make one call and return what it
# launched as [[kernel with its template arguments, splits (grid z), threads]]
PRELUDE = """
import ctypes, json, sys
sys.path.insert(0, {root!r})
fake = ctypes.CDLL({stub!r}, mode=ctypes.RTLD_GLOBAL)
fake.fake_launches.restype = ctypes.c_char_p
fake.fake_allocated.restype = ctypes.c_size_t
fake.fake_memory.argtypes = [ctypes.c_size_t]
from xtc_amd.runtimes.hip import capi
L = capi.lib()
assert L.xtc_hip_init(0) == 0, capi.last_error()
out = []

def launched():
    rows = []
    for line in fake.fake_launches().decode().splitlines():
        name, grid, threads = line.split("|")
        for noise in ("void ", "xtc_hip::", "(anonymous namespace)::"):
            name = name.replace(noise, "")
        name = name.split("(")[0]
        rows.append([name, int(grid.split()[2]), int(threads)])
    return rows

def matmul(dtype, M, N, K, tile=None, split=0, fn="xtc_hip_matmul", a=256, b=256, **kw):
    d = capi.MatmulDesc(dtype=capi.DTYPE_IDS[dtype], M=M, N=N, K=K, split_k=split, xcd_remap=1, **kw)
    if tile:
        d.tile = capi.Tile(*tile)
    p = ctypes.c_void_p
    rc = getattr(L, fn)(ctypes.byref(d), p(a), p(b), p(256), None)
    return capi.last_error() if rc else launched()

def conv(dtype, n, h, w, c, f, r, s, stride=1, pad=0, tile=None, split=0):
    d = capi.Conv2dDesc(dtype=capi.DTYPE_IDS[dtype], N=n, H=h, W=w, C=c, F=f, R=r, S=s, stride_h=stride,
                        stride_w=stride, pad_top=pad, pad_bottom=pad, pad_left=pad, pad_right=pad, split_k=split)
    if tile:
        d.tile = capi.Tile(*tile)
    p = ctypes.c_void_p
    rc = L.xtc_hip_conv2d(ctypes.byref(d), p(256), p(256), p(256), None)
    return capi.last_error() if rc else launched()
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    """run(script): what the script appended to `out`, in a process of its own."""
    stub = tmp_path_factory.mktemp("hip_stub") / "libfake_hip.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-shared", "-fPIC", "-I/opt/rocm/include",
                    str(ROOT / "tests" / "hip_stub" / "fake_hip.cpp"), "-o", str(stub)], check=True)
    prelude = PRELUDE.format(root=str(ROOT), stub=str(stub))

    def go(script: str):
        code = prelude + script + "\nprint('@' + json.dumps(out))\n"
        res = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=120)
        assert res.returncode == 0, res.stderr
        return json.loads(res.stdout.split("@")[-1])

    return go


def test_captured_calls_without_whole_vectors_take_no_scratch(run):
    # eager calls split K and leave the stream's workspace behind; a captured
    # one must not keep its address: a later, larger call frees it
    eager, captured, conv_eager, conv_captured, after, noalloc = run("""
out.append(matmul("float32", 509, 1021, 777))
fake.fake_capturing(1)
out.append(matmul("float32", 509, 1021, 777))
fake.fake_capturing(0)
out.append(conv("float32", 1, 14, 14, 333, 66, 3, 3, pad=1, split=4))
fake.fake_capturing(1)
out.append(conv("float32", 1, 14, 14, 333, 66, 3, 3, pad=1, split=4))
fake.fake_capturing(0)
out.append(matmul("float32", 509, 1021, 777))
fake.fake_capturing(1)
out.append(matmul("float32", 509, 1021, 777, fn="xtc_hip_matmul_noalloc"))
""")
    kernel = "gemm_planes<float, 64, 64, 32, 2, 2, false, false, false, 1, 1>"
    assert eager[-1] == [kernel, 4, 256] and after == eager[-1:]
    assert captured == [[kernel, 1, 256]]
    assert conv_eager[-1][1] == 4 and conv_captured == [[conv_eager[-1][0], 1, conv_eager[-1][2]]]
    # the static scratch of the no-allocation entry point stays: split as ever
    assert noalloc[-1] == [kernel, 4, 256]


def test_calls_without_whole_vectors_run_unsplit_where_scratch_cannot_be_had(run):
    # no memory at all, and enough for the partial sums but not the counters;
    # a conv whose filters are not whole vectors; then memory again
    none, counters, conv, later, message = run("""
fake.fake_memory(1 << 20)
out.append(matmul("float32", 509, 1021, 777))
fake.fake_memory(4 * 509 * 1024 * 4 + 1000)
out.append(matmul("float32", 509, 1021, 777))
fake.fake_memory(1000)
out.append(conv("bfloat16", 1, 14, 14, 333, 67, 3, 3, pad=1, split=4))
fake.fake_memory(1 << 30)
out.append(matmul("float32", 509, 1021, 777))
out.append(L.xtc_hip_last_error().decode())
""")
    kernel = "gemm_planes<float, 64, 64, 32, 2, 2, false, false, false, 1, 1>"
    assert none == counters == [[kernel, 1, 256]]
    assert conv == [["gemm_planes<__bf16, 64, 64, 64, 2, 2, true, false, false, 1, 1>", 1, 256]]
    assert later[-1] == [kernel, 4, 256]
    assert message == ""


@pytest.mark.parametrize("shape,split,trans_a,splits", [
    ((509, 1021, 777), 4, 0, 4),
    ((4097, 4097, 300), 2, 0, 1),  # 134 MB of partial sums
    ((2500, 1001, 4001), 3, 1, 1),  # 30 MB of them behind a 40 MB copy of A
    ((2500, 1001, 2001), 3, 1, 3),
])
def test_both_entry_points_split_ragged_calls_alike(run, shape, split, trans_a, splits):
    # the partial sums of either entry point stay within the static scratch,
    # so that the sums are taken in the same order
    M, N, K = shape
    grown, static = run(f"""
for fn in ("xtc_hip_matmul", "xtc_hip_matmul_noalloc"):
    out.append(matmul("float32", {M}, {N}, {K}, split={split}, trans_a={trans_a}, tile=(64, 64, 32, 2, 2), fn=fn))
""")
    kernel = "gemm_planes<float, 64, 64, 32, 2, 2, false, false, false, 1, 1>"
    assert grown[-1] == static[-1] == [kernel, splits, 256]
