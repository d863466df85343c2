# SPDX-License-Identifier: BSD-3-Clause
"""Index arithmetic of the pad and crop kernel (xtc_amd/csrc/row_copy.hpp), on
the CPU, where its 32-bit indices end: innermost extents up to 2^31 - 1.  Each
group of four is compared, element by element, with the same element computed
in 64 bits (Python integers): where it lies in the output, whether it is
written, and which input element, if any, it is read from."""

from __future__ import annotations

import shutil
import subprocess
from math import prod
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "xtc_amd" / "csrc"

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")

# stdin: pad outer, `outer` times (out in before), out_len in_len shift, then
# group numbers; stdout per group: its four elements as "row col written
# inside src_row src_col"
HARNESS = r"""
#define __host__
#define __device__
#include "row_copy.hpp"
#include <cstdio>
using namespace xtc_hip;
int main() {
  int pad, n;
  RowCopyDims d = {};
  if (scanf("%d %d", &pad, &d.outer) != 2) return 1;
  for (int k = 0; k < d.outer; ++k)
    if (scanf("%u %u %u", &d.out_shape[k], &d.in_shape[k], &d.before[k]) != 3) return 1;
  if (scanf("%u %u %u", &d.out_len, &d.in_len, &d.shift) != 3) return 1;
  d.groups = (d.out_len + 3) / 4;
  unsigned i;
  while (scanf("%u", &i) == 1) {
    const RowGroup g = pad ? row_group<true>(d, i) : row_group<false>(d, i);
    const bool in4 = row_has4(g.c, d.in_len), out4 = row_has4(g.col, d.out_len);
    for (unsigned e = 0; e < 4; ++e)
      printf("%u %lld %d %d %u %lld\n", g.row, (long long)g.col + e,
             out4 || (e < 3 && row_has(g.col, e, d.out_len)), g.inside && (in4 || row_has(g.c, e, d.in_len)),
             g.src_row, (long long)(int)g.c + e);
  }
  return 0;
}
"""


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("row_copy")
    (tmp / "h.cpp").write_text(HARNESS)
    subprocess.run(["g++", "-std=c++17", "-O1", "-fsanitize=undefined", "-fno-sanitize-recover=all", f"-I{CSRC}",
                    str(tmp / "h.cpp"), "-o", str(tmp / "h")], check=True)
    return tmp / "h"


TOP = 2**31 - 1
# (pad?, input shape, [(before, after)])
CASES = [
    *[(True, (n - b - a,), [(b, a)]) for n in range(TOP - 4, TOP + 1) for b, a in ((0, 1), (1, 0), (3, 2), (TOP - 9, 0))],
    *[(False, (n,), [(b, a)]) for n in range(TOP - 4, TOP + 1) for b, a in ((0, 1), (1, 0), (3, 2), (n - 3, 0), (n - 5, 1))],
    (True, (2, 5), [(1, 2), (3, TOP // 5 - 20)]),
    (True, (0, 6), [(2, 1), (1, 1)]),
    (True, (4, 0), [(0, 0), (2, 3)]),
    (True, (3, 1, 2, 9), [(1, 1), (0, 3), (1, 0), (5, 2)]),
    (False, (5, 4, 3, 16), [(1, 1), (0, 3), (1, 0), (5, 2)]),
]


@pytest.mark.parametrize("pad,shape,pads", CASES)
def test_groups_against_64_bit_indices(harness, pad, shape, pads):
    sign = 1 if pad else -1
    out = [s + sign * (b + a) for s, (b, a) in zip(shape, pads)]
    groups = (out[-1] + 3) // 4
    total = prod(out[:-1]) * groups
    assert prod(out) <= TOP
    near = {0, 1, groups - 1, groups, total - 2, total - 1, pads[-1][0] // 4, (pads[-1][0] + shape[-1]) // 4}
    picked = sorted(i for i in (near | set(range(min(total, 64)))) if 0 <= i < total)
    lines = [f"{int(pad)} {len(shape) - 1}"]
    lines += [f"{o} {s} {b}" for o, s, (b, _) in zip(out[:-1], shape[:-1], pads[:-1])]
    lines += [f"{out[-1]} {shape[-1]} {pads[-1][0]}", *map(str, picked)]
    got = subprocess.run([str(harness)], input="\n".join(lines), capture_output=True, text=True, check=True).stdout
    rows = iter(got.splitlines())
    for i in picked:
        for e in range(4):
            row, col, written, read, src_row, src_col = map(int, next(rows).split())
            assert (row, col) == (i // groups, 4 * (i % groups) + e)
            assert written == (col < out[-1]), (i, e)
            if not written:
                continue
            rem, src = row, [col - sign * pads[-1][0]]
            for o, (b, _) in zip(out[-2::-1], pads[-2::-1]):
                src.insert(0, rem % o - sign * b)
                rem //= o
            want_read = all(0 <= s < n for s, n in zip(src, shape))
            assert read == want_read, (i, e)
            if want_read:
                flat = 0
                for s, n in zip(src[:-1], shape[:-1]):
                    flat = flat * n + s
                assert (src_row, src_col) == (flat, src[-1]), (i, e)
