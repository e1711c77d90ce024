"""How a backward call cuts its long rows and columns (plan_segments, device_common.h), on the CPU: every work item of a
plan and every place of its partial sums, whatever lengths the caller gives."""
from __future__ import annotations

import ctypes as C
import os
import random
import shutil
import subprocess

import pytest

from test_kernel_resources import CSRC, HIPCC

pytestmark = pytest.mark.skipif(shutil.which(HIPCC) is None, reason="hipcc not installed")
SEGMENTS = 16
SOURCE = """
#include "bwd_scratch.h"
using namespace dk;
extern "C" int plan(const int32_t *lengths, int rows, int per_step, int64_t copies, int slots, double limit, double share, int heads,
                    int32_t *n, int32_t *out) {
  const SegView s = plan_segments(lengths, rows, per_step, copies, slots, limit, share, heads);
  for (int i = 0; i < kMaxSegments; ++i) n[i] = s.n[i];
  out[0] = s.entries, out[1] = s.slots, out[2] = (int)segment_items(s, rows);
  return kMaxSegments;
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = str(tmp_path_factory.mktemp("plan"))
    with open(os.path.join(d, "plan.hip"), "w") as f:
        f.write(SOURCE)
    subprocess.run([HIPCC, "--cuda-host-only", "-x", "hip", "-O1", "-std=c++17", "-fPIC", "-shared", "-I", CSRC, os.path.join(d, "plan.hip"),
                    "-o", os.path.join(d, "plan.so")], check=True, capture_output=True)
    lib = C.CDLL(os.path.join(d, "plan.so"))

    def run(lengths, per_step, copies, slots, limit, share, heads):
        n, out = (C.c_int32 * SEGMENTS)(), (C.c_int32 * 3)()
        assert lib.plan((C.c_int32 * len(lengths))(*lengths), len(lengths), per_step, C.c_int64(copies), slots, C.c_double(limit),
                        C.c_double(share), heads, n, out) == SEGMENTS
        return list(n), *out

    return run


def _segments(length, per_step, heads, entries):  # of a row, as the kernels count them before the limit by its place
    steps = -(-length // per_step) * heads
    return max(1, (2 * steps + entries) // (2 * entries))


@pytest.mark.parametrize("order", ["descending", "ascending", "random", "one long at the end", "any"])
@pytest.mark.parametrize("per_step,heads", [(1, 1), (2, 1), (1, 4)])
def test_places_of_any_lengths(plan, order, per_step, heads):
    rng = random.Random(order)
    cut = 0
    for rows in (1, 2, 23, 47, 128, 300):
        for slots in (256, 768):
            lengths = [rng.choice((1, 4, 9, rng.randint(0, 400))) for _ in range(rows)]
            if order == "descending":
                lengths.sort(reverse=True)
            elif order == "ascending":
                lengths.sort()
            elif order == "one long at the end":
                lengths = [3] * (rows - 1) + [400]
            elif order == "any":  # nonsense from the caller
                lengths = [rng.choice((-5, 0, 7, 2**31 - 1, -2**31, rng.randint(0, 500))) for _ in range(rows)]
            n, entries, places, items = plan(lengths, per_step, 8, slots, 1.0, 0.6, heads)
            if not entries:
                assert not any(n) and not places and items == rows
                continue
            cut += 1
            assert all(a >= b for a, b in zip(n[1:], n[2:])) and n[1] <= rows and items == rows + sum(n[1:])
            # what the launch does with each row, of the length it has (the plan's or any other): segment s of the row at
            # `place` leaves its sum at s * n[1] + place
            for place in range(rows):
                most = 1 + sum(place < x for x in n[1:])
                real = lengths[place] if order != "any" else rng.randint(0, 10**6)
                for seg in range(min(_segments(real, per_step, heads, entries), most)):
                    assert seg * n[1] + place < places or most == 1, (rows, place, seg, n, places)
                if order != "any":  # ... and every row gets the segments that its length asks for
                    assert _segments(real, per_step, heads, entries) <= most
    assert cut >= 3
