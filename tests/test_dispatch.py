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

def conv(dtype, n, h, w, c, f, r, s, stride=1, pad=0, tile=None, split=0, pad_value=0.0):
    d = capi.Conv2dDesc(dtype=capi.DTYPE_IDS[dtype], N=n, H=h, W=w, C=c, F=f, R=r, S=s, stride_h=stride,
                        stride_w=stride, pad_top=pad, pad_bottom=pad, pad_left=pad, pad_right=pad, split_k=split, pad_value=pad_value)
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


@pytest.mark.parametrize("shape,splits,static_splits", [
    ((2500, 1001, 4001), 3, 1),  # 30 MB of partial sums beside a 40 MB copy of A
    ((2900, 429, 7572), 4, None),  # an 88 MB copy, which the static scratch refuses
])
def test_copies_of_transposed_operands_cost_growing_calls_no_split(run, shape, splits, static_splits):
    M, N, K = shape
    grown, static = run(f"""
for fn in ("xtc_hip_matmul", "xtc_hip_matmul_noalloc"):
    out.append(matmul("float32", {M}, {N}, {K}, split={splits}, trans_a=1, tile=(64, 64, 32, 2, 2), fn=fn))
""")
    kernel = "gemm_planes<float, 64, 64, 32, 2, 2, false, false, false, 1, 1>"
    assert grown[-1] == [kernel, splits, 256]
    assert static[-1] == [kernel, static_splits, 256] if static_splits else "scratch" in static


@pytest.mark.parametrize("dtype,tile,split,shape,trans_b,kernel", [
    ("float32", (64, 64, 32, 2, 2), 2, (2000, 2304, 2600), 0, "gemm_planes<float, 64, 64, 32, 2, 2, false, false, true, 1, 1>"),
    ("float32", (64, 64, 32, 2, 2), 1, (2048, 2048, 1024), 1, "gemm_planes<float, 64, 64, 32, 2, 2, false, true, true, 1, 1>"),
    ("float32", (64, 64, 32, 2, 2), 8, (1000, 1104, 1200), 0, "gemm_planes<float, 64, 64, 32, 2, 2, false, false, true, 1, 1>"),
    ("float32", (64, 64, 32, 2, 2), 8, (768, 768, 4096), 0, "gemm_planes<float, 64, 64, 32, 2, 2, false, false, true, 1, 1>"),
    ("float32", (128, 128, 32, 2, 2), 1, (3000, 3000, 3000), 0, "gemm_kernel<float, 128, 128, 32, 2, 2, false, 1>"),
    ("float32", (128, 128, 32, 2, 2), 3, (256, 4608, 8192), 0, "gemm_kernel<float, 128, 128, 32, 2, 2, false, 1>"),
    ("float32", (128, 256, 32, 2, 4), 2, (2048, 1024, 4096), 0, "gemm_planes<float, 128, 256, 32, 2, 4, false, false, true, 1, 1>"),
    ("bfloat16", (128, 128, 64, 2, 2), 4, (256, 8192, 4608), 0, "gemm_planes<__bf16, 128, 128, 64, 2, 4, false, false, true, 2, 1>"),
    ("bfloat16", (128, 128, 64, 2, 2), 2, (256, 8192, 4608), 0, "gemm_planes<__bf16, 128, 128, 64, 2, 4, false, false, true, 1, 2>"),
    ("bfloat16", (128, 128, 64, 2, 2), 4, (256, 4608, 8192), 1, "gemm_planes<__bf16, 128, 128, 64, 2, 4, false, true, true, 1, 1>"),
])
def test_named_matmuls_run_their_tile_and_split(run, dtype, tile, split, shape, trans_b, kernel):
    M, N, K = shape
    (rows,) = run(f"out.append(matmul({dtype!r}, {M}, {N}, {K}, tile={tile}, split={split}, trans_b={trans_b}))")
    assert [rows[-1][0], rows[-1][1]] == [kernel, split]


@pytest.mark.parametrize("tile,split,shape", [((128, 64, 64, 2, 2), 4, (1, 34, 34, 256, 512, 3)),
                                              ((128, 128, 64, 2, 2), 8, (1, 17, 17, 1024, 1024, 3))])
def test_named_convs_run_their_split(run, tile, split, shape):
    n, h, w, c, f, r = shape
    (rows,) = run(f"out.append(conv('bfloat16', {n}, {h}, {w}, {c}, {f}, {r}, {r}, pad=1, tile={tile}, split={split}))")
    assert rows[-1][0].startswith(f"gemm_planes<__bf16, {tile[0]}, {tile[1]}, 64,") and rows[-1][1] == split


def test_split_wave_depths_behind_the_64x64_tile(run):
    # 512^3 at split 4: the tile's depths 4 (the default) and 2 are the split-wave kernel's ring
    rows = run("""
for stages in (0, 4, 2):
    out.append(matmul("float32", 512, 512, 512, tile=(64, 64, 32, 2, 2), split=4, stages=stages))
""")
    assert [r[-1][0] for r in rows] == [f"gemm_f32_splitwave<4, {depth}>" for depth in (4, 4, 2)]


def test_explorer_points_are_kernels_of_their_own(run):
    # every sample of the explorer's space launches something else: a depth that
    # only renames the one pipeline of gemm_planes is no point
    points, launches = run("""
import xtc_amd.graphs.xtc.op as O
from xtc_amd.search.strategies import Strategies
a, b = O.tensor((1024, 1024), "float32", name="A"), O.tensor((1024, 1024), "float32", name="B")
with O.graph(name="mm") as gb:
    O.matmul(a, b, name="C")
wide = [x for x in Strategies.create("tile_hip", gb.graph)._points()
        if (x[0], x[2], x[4]) in ((256, 128, 32), (128, 256, 32), (128, 128, 32), (64, 64, 32))]
out.append([tuple(x) for x in wide])
out.append([matmul("float32", 1024, 1024, 1024, tile=(x[0], x[2], x[4], x[0] // x[1], x[2] // x[3]), split=x[5],
                   stages=x[6])[-1] for x in wide])
""")
    assert len(points) > 20
    kernels = [tuple(x) + tuple(p[:6]) for p, x in zip(points, launches)]
    assert len(set(kernels)) == len(kernels)


@pytest.mark.parametrize("dtype,tile,pad_value,launches", [
    # by default and on the gather's own tiles in place, else on whole-vector copies
    ("float32", None, 0.0, ["gemm_planes<float, 128, 64, 32, 4, 2, true, false, false, 1, 1>"]),
    ("float32", (128, 64, 32, 4, 2), 0.0, ["gemm_planes<float, 128, 64, 32, 4, 2, true, false, false, 1, 1>"]),
    ("float32", (64, 64, 32, 2, 2), 0.0, ["gemm_planes<float, 64, 64, 32, 2, 2, true, false, false, 1, 1>"]),
    ("float32", (64, 64, 16, 2, 2), 0.0, ["pad_channels_kernel<float>"] * 2 + ["gemm_kernel<float, 64, 64, 16, 2, 2, true, 1>"]),
    ("float32", (128, 64, 32, 2, 2), 0.0, ["pad_channels_kernel<float>"] * 2 + ["gemm_kernel<float, 128, 64, 32, 2, 2, true, 1>"]),
    ("bfloat16", None, 0.0, ["gemm_planes<__bf16, 64, 64, 64, 2, 2, true, false, false, 1, 1>"]),
    ("bfloat16", (32, 64, 32, 1, 2), 0.0, ["pad_channels_kernel<unsigned short>"] * 2 + ["gemm_kernel<__bf16, 32, 64, 32, 1, 2, true, 1>"]),
    # an infinite pad value cannot be copied beside zero channels: any tile is gathered
    ("float32", (32, 32, 16, 1, 1), float("inf"), ["gemm_planes<float, 128, 64, 32, 4, 2, true, false, false, 1, 1>"]),
])
def test_named_convs_without_whole_vectors_run_their_tile(run, dtype, tile, pad_value, launches):
    pad_value = f"float('{pad_value}')"
    (rows,) = run(f"out.append(conv({dtype!r}, 4, 224, 224, 3, 64, 7, 7, stride=2, pad=3, tile={tile}, split=1, "
                  f"pad_value={pad_value}))")
    assert [r[0] for r in rows] == launches


def test_default_conv_sample_of_the_explorer_maps_on_the_gather():
    import xtc_amd.graphs.xtc.op as O
    from xtc_amd.backends.hip import Backend
    from xtc_amd.search.strategies import Strategies

    x, w = O.tensor((4, 224, 224, 3), "float32", name="I"), O.tensor((7, 7, 3, 64), "float32", name="W")
    with O.graph(name="stem") as gb:
        O.conv2d(x, w, stride=(2, 2), name="C")
    backend, strategy = Backend(gb.graph), Strategies.create("tile_hip", gb.graph)
    sch = backend.get_scheduler()
    strategy.generate(sch, strategy.default_schedule())
    compiler = backend.get_compiler(schedule_policy="strict")
    tiles = [compiler.kernel_configs(s.schedule())["C"].tile for s in (sch, backend.get_scheduler())]
    assert tiles == [(128, 64, 32, 4, 2)] * 2


def test_default_queries_name_what_an_unnamed_call_runs(run):
    # over shapes, layouts and strides: the tile and split that the query
    # returns, named, launch what the zeroed tile does
    pairs = run("""
import random
rng = random.Random(3)
pick = lambda step: max(step, int(8 * 1024 ** rng.random()) // step * step)
for i in range(400):
    dtype, step = rng.choice(("float32", "bfloat16", "float64")), rng.choice((1, 8, 64, 128))
    M, N, K = pick(rng.choice((1, 64))), pick(step), pick(step)
    kw = dict(trans_b=rng.randint(0, 1), trans_a=int(rng.random() < 0.2), relu=rng.randint(0, 1))
    if rng.random() < 0.2:
        kw["ldb"] = (K if kw["trans_b"] else N) + rng.choice((1, 8, 64))
    d = capi.MatmulDesc(dtype=capi.DTYPE_IDS[dtype], M=M, N=N, K=K, **kw)
    tile, split = capi.matmul_default_tile(d)
    out.append([repr((dtype, M, N, K, kw)), matmul(dtype, M, N, K, **kw),
                matmul(dtype, M, N, K, tile=tile, split=split, **kw)])
for i in range(200):
    dtype, r = rng.choice(("float32", "bfloat16", "float64")), rng.choice((1, 3, 5))
    h, c, f = rng.randint(7, 60), rng.choice((3, 16, 32, 64, 256)), rng.choice((7, 16, 64, 96, 512))
    d = capi.Conv2dDesc(dtype=capi.DTYPE_IDS[dtype], N=1, H=h, W=h, C=c, F=f, R=r, S=r, stride_h=1, stride_w=1,
                        pad_top=1, pad_bottom=1, pad_left=1, pad_right=1)
    tile, split = capi.conv2d_default_tile(d)
    out.append([repr((dtype, h, c, f, r)), conv(dtype, 1, h, h, c, f, r, r, pad=1),
                conv(dtype, 1, h, h, c, f, r, r, pad=1, tile=tile, split=split)])
""")
    assert len(pairs) == 600
    for what, unnamed, named in pairs:
        assert isinstance(named, list), (what, named)
        # but for counters cleared when they are first allocated
        unnamed, named = ([r for r in rows if r[0] != "fill_zero_kernel"] for rows in (unnamed, named))
        assert unnamed == named, what


def test_default_configs_report_the_kernel_that_runs():
    import xtc_amd.graphs.xtc.op as O
    from xtc_amd.backends.hip import Backend

    a, b = O.tensor((2048, 1024), "float32", name="A"), O.tensor((1024, 2048), "float32", name="B")
    with O.graph(name="mm") as gb:
        O.matmul(a, b, name="C")
    backend = Backend(gb.graph)
    cfg = backend.get_compiler().kernel_configs(backend.get_scheduler().schedule())["C"]
    assert cfg.tile == (128, 128, 32, 2, 4) and cfg.split_k == 1 and cfg.source == "default"


@pytest.mark.parametrize("cut,tile", [(2048, (256, 128, 32, 4, 2)), (2, (128, 128, 32, 2, 2))])
def test_default_pieces_of_a_split_see_their_alignment(cut, tile):
    # 2048 columns from `cut` on: whole vectors, or B rows that start 8 bytes past one
    import xtc_amd.graphs.xtc.op as O
    from xtc_amd.backends.hip import Backend

    a, b = O.tensor((3000, 1024), "float32", name="A"), O.tensor((1024, 4104), "float32", name="B")
    with O.graph(name="mm") as gb:
        O.matmul(a, b, name="C")
    backend = Backend(gb.graph)
    sch = backend.get_scheduler()
    sch.split("j", {"l": 0, "m": cut, "r": cut + 2048})
    pieces = backend.get_compiler().kernel_configs(sch.schedule())["C"].pieces
    assert (pieces[1].n0, pieces[1].N) == (cut, 2048)
    assert pieces[1].config.tile == tile and pieces[1].config.source == "default"
