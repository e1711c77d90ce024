"""How a backward call cuts its long rows and columns (plan_segments, device_common.h), on the CPU: every work item of a
plan and every place of its partial sums, whatever lengths the caller gives."""
from __future__ import annotations

import array
import copy
import ctypes as C
import os
import pickle
import random
import shutil
import subprocess

import numpy as np
import pytest
import torch

from dkernel_amd import LocalStrideSparseAttention, SparseAttention, _lib
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
// 16-bit pass at the 128-wide tile: out = {partials per q head?, entries per segment of dQ and of dK / dV}
extern "C" void scratch(int batch, int Hq, int Hkv, int D, int queries, int keys, int rows, int cols, const int32_t *pair_lengths,
                        const int32_t *col_lengths, int32_t *out) {
  BwdParams p;
  p.seqs = SeqView{batch, queries, keys, 0};
  p.Hq = Hq, p.Hkv = Hkv, p.D = D;
  p.csr = LutView{nullptr, nullptr, 0, 0, 1, 1, rows, 64, 64, Hq, 0, 0};
  p.csc = LutView{nullptr, nullptr, 0, 0, 1, 1, cols, 64, 64, Hq, 0, 0};
  p.csr.pair_lengths = pair_lengths, p.csc.row_lengths = col_lengths;
  const size_t group = Hq == Hkv ? 0 : 2 * (size_t)batch * Hq * keys * D * 4;
  const BwdScratch s = plan_bwd_scratch(p, group, 512, true, 512, kWalkFrom, kLeastGain);
  out[0] = s.group > 0, out[1] = s.dq.entries, out[2] = s.kv.entries;
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

    def scratch(batch, Hq, Hkv, D, L, rows, cols, pairs, columns):
        out = (C.c_int32 * 3)()
        at = [None if x is None else C.c_void_p(x.buffer_info()[0] + 4 * skip) for x, skip in ((pairs, rows), (columns, 0))]
        lib.scratch(batch, Hq, Hkv, D, L, L, rows, cols, *at, out)
        return list(out)

    def run(lengths, per_step, copies, slots, limit, share, heads):
        n, out = (C.c_int32 * SEGMENTS)(), (C.c_int32 * 3)()
        assert lib.plan((C.c_int32 * len(lengths))(*lengths), len(lengths), per_step, C.c_int64(copies), slots, C.c_double(limit),
                        C.c_double(share), heads, n, out) == SEGMENTS
        return list(n), *out

    run.scratch = scratch
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


def _lengths(mask, first, last, limit, order, pairs):
    """Straight from the pattern (heads, rows, columns): entries of the rows first .. last at columns below `limit`."""
    heads, rows, _ = mask.shape
    inside = (np.arange(rows) >= first) & (np.arange(rows) <= last)
    lens = mask[:, :, :limit].sum(2) * inside
    if pairs:
        pad = rows % 2
        lens = np.pad(lens, ((0, 0), (0, pad))).reshape(heads, -1, 2).sum(2)
        inside = np.pad(inside, (0, pad)).reshape(-1, 2).any(1)
    lens = np.where(inside[None], lens, -1)
    return np.take_along_axis(lens, order, axis=1).max(0).tolist()


def _global_mask(heads, n):
    i = np.arange(n)
    mask = np.repeat((np.abs(i[:, None] - i[None]) <= 1)[None], heads, axis=0)
    mask |= np.random.default_rng(n).random((heads, n, n)) < 0.05
    mask[:, :2] = True
    mask[:, :, :2] = True
    mask[heads - 1, n // 2] = True
    return mask


@pytest.mark.parametrize("block", [16, 32, 64, 128])
@pytest.mark.parametrize("heads,n,causal", [(1, 16, False), (3, 24, False), (4, 24, True)])
def test_lengths_of_a_call(heads, n, causal, block):
    mask = _global_mask(heads, n)
    if causal:
        mask = mask & np.tril(np.ones((n, n), dtype=bool))
        mask[:, n // 3] = np.arange(n) <= n // 3
    mod = SparseAttention(block, torch.from_numpy(mask), causal=causal)
    tiles = np.zeros((heads, n * block // 64, n * block // 64), dtype=bool)  # 64 x 64 tiles with an attended block
    for h, i, j in zip(*np.nonzero(mask)):
        tiles[h, i * block // 64:max(i * block // 64 + 1, (i + 1) * block // 64), j * block // 64:max(j * block // 64 + 1, (j + 1) * block // 64)] = True
    if causal:
        tiles &= np.tril(np.ones(tiles.shape[1:], dtype=bool))
    tables = mod.kwargs["row_lengths"][-1]
    csr, csc = tables.csr, tables.csc
    assert (csr is None) == (not mod.kwargs["unsorted_rows"])
    rows, step = tiles.shape[1], mod.lut_group
    for first, last, keys in [(0, rows - 1, rows - 1), (0, 0, 0), (0, 1, 1), (1, 2, 2), (1, rows - 2, rows - 1), (2, 2, 2), (0, rows // 2, rows // 2)]:
        for table, mask_t, call in ((csr, tiles, (first, last, 2**31 - 1)), (csc, tiles.transpose(0, 2, 1), (0, keys, last + 1))):
            if table is None:
                continue
            got, order = table.of_call(*call).tolist(), table.order.numpy().astype(np.int64)
            lens = mask_t[::step].sum(2)
            assert (np.sort(order[:, :rows], axis=1) == np.arange(rows)).all()
            assert (np.diff(np.take_along_axis(lens, order[:, :rows], axis=1)) <= 0).all()
            limit = min(call[2], rows)
            assert got[:rows] == _lengths(mask_t[::step], call[0], call[1], limit, order[:, :rows], False)
            assert got[rows:] == _lengths(mask_t[::step], call[0], call[1], limit, order[:, rows:], True)


def test_lengths_refuse_what_they_cannot_read():
    ptr, idx, out = (C.c_int32 * 4)(0, 1, 2, 3), (C.c_int32 * 3)(0, 1, 2), (C.c_int32 * 5)()

    def call(order, at=ptr, heads=1):
        return _lib.lib().dk_call_row_lengths(at, idx, (C.c_int32 * 5)(*order), heads, 3, 3, 0, 2, 2, out)

    assert call((2, 1, 0, 1, 0)) == 0 and list(out) == [0, 1, 1, 0, 2]
    for bad in ((3, 1, 0, 1, 0), (-1, 1, 0, 1, 0), (2, 1, 0, 2, 0)):
        assert call(bad) != 0
    assert call((2, 1, 0, 1, 0), at=None) != 0 and call((2, 1, 0, 1, 0), heads=0) != 0


def _plan_of(plan, mod, batch, Hq, Hkv, D, L):
    tables = mod.kwargs["row_lengths"][0]
    rows = tables.csc.rows
    lengths, pairs, columns = tables.of_call(0, L, L)
    assert lengths.csc_rows == columns.buffer_info()[0] and not lengths.csr_rows
    how = plan.scratch(batch, Hq, Hkv, D, L, rows, rows, pairs, columns)
    inside = sorted(x for x in columns[:rows] if x >= 0)
    return how, inside


@pytest.mark.parametrize("batch,heads,kv_heads,L,tables", [
    (1, 32, 8, 2048, (2048, 8192, 32768)), (1, 32, 8, 4096, (4096, 8192, 32768)), (4, 32, 8, 2048, (2048, 8192, 32768)),
    (1, 32, 8, 1000, (1000, 8192)), (1, 8, 8, 3000, (3000, 16384)), (1, 16, 4, 8000, (8000, 32768)), (2, 12, 12, 300, (300, 8192))])
def test_the_plan_of_a_call_does_not_depend_on_the_tables_length(plan, batch, heads, kv_heads, L, tables):
    want = None
    for table in tables:
        mod = LocalStrideSparseAttention(heads, table, 64, 16, 8, num_kv_heads=kv_heads)
        # (the most over the heads at each place: a few per cent more in a longer table, whose heads list the call's columns at other places)
        how, inside = _plan_of(plan, mod, batch, heads, kv_heads, 128, L)
        want = want or (how, inside)
        assert how[0] == want[0][0], (table, how, want)  # walks whole groups, or not
        assert (how[2] > 0) == (want[0][2] > 0) and abs(how[2] - want[0][2]) <= max(1, 0.05 * want[0][2]), (table, how, want)
    if (batch, heads, L) == (1, 32, 2048):
        assert want[0][0] == 1  # one workgroup per q head: 28 steps a slot are no work for whole groups
    if (batch, heads, L) == (4, 32, 2048):
        assert want[0][0] == 0


@pytest.mark.parametrize("saved", [None, ((array.array("i", [3, 2, 5]), array.array("i", [2, 2, 4])),)])
def test_modules_saved_with_other_lengths_get_the_present_ones(saved):
    mod = SparseAttention(32, torch.from_numpy(_global_mask(2, 20)), causal=False)
    mod.kwargs["row_lengths"][0].of_call(0, 65, 65)
    old = copy.deepcopy(mod)
    assert old.kwargs == mod.kwargs and not old.kwargs["row_lengths"][0]._calls
    if saved is None:
        del old.kwargs["row_lengths"]
    else:
        old.kwargs["row_lengths"] = saved
    assert pickle.loads(pickle.dumps(old)).kwargs == mod.kwargs


@pytest.mark.parametrize("batch,heads,L,local,vert,cut", [
    (2, 16, 1831, 16, 8, False), (1, 32, 1377, 16, 8, False), (2, 16, 1333, 8, 4, False),   # the longest column hardly stands out
    (2, 8, 1464, 16, 8, False),                                                              # or too much is cut with it
    (1, 8, 3181, 4, 16, True), (2, 12, 2776, 4, 16, True), (1, 16, 8546, 16, 8, True), (1, 12, 4872, 8, 8, True)])
def test_columns_are_cut_where_it_gains(plan, batch, heads, L, local, vert, cut):
    mod = LocalStrideSparseAttention(heads, L, 64, local, vert)
    how, _ = _plan_of(plan, mod, batch, heads, heads, 128, L)
    assert (how[2] > 0) == cut, how
