"""Masked 64 x 64 tiles (pattern blocks of 16 and 32): the kernels multiply 32 x 32 quadrants and leave out those
that hold no attended block.  Sparse random patterns, in which most tiles hold one or two quadrants and single
16-token blocks inside them, at every tile width, forward and backward, against the fp32 oracle at the 16-bit bar.
(The first six forwards are split along the keys, the others run single rows; row pairs and head groups:
test_gpu_large_launch_kernels.py.)"""
import math

import numpy as np
import pytest
import torch

from dkernel_amd import SparseAttention, ops
from helpers import LSE_TOL, TOL, assert_close, make_qkv, oracle_fwd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,L,D,bs,dtype,causal,density", [
    (1, 2, 2, 700, 128, 32, torch.bfloat16, True, 0.06),
    (1, 2, 2, 650, 128, 16, torch.float16, True, 0.02),
    (2, 4, 1, 513, 64, 32, torch.float16, False, 0.05),
    (1, 4, 1, 400, 64, 16, torch.bfloat16, False, 0.03),
    (1, 2, 1, 450, 256, 32, torch.bfloat16, True, 0.08),
    (1, 2, 2, 330, 200, 16, torch.bfloat16, True, 0.04),
    (1, 3, 3, 575, 96, 32, torch.bfloat16, False, 0.05),
    (1, 4, 4, 2600, 120, 32, torch.float16, True, 0.03),   # (single rows, and so are the cases below)
    (1, 8, 8, 2100, 128, 32, torch.bfloat16, True, 0.03),
    (4, 32, 32, 400, 128, 16, torch.bfloat16, False, 0.05),
    (1, 2, 2, 650, 64, 32, torch.float16, "global", 0.05),   # (whole tiles)
    (2, 2, 2, 450, 40, 16, torch.bfloat16, "global", 0.03),
    (1, 2, 2, 650, 128, 32, torch.bfloat16, "global", 0.05),
])
def test_sparse_tiles(B, Hq, Hkv, L, D, bs, dtype, causal, density):
    long_rows, causal = causal == "global", causal is True
    print(f"case B={B} Hq={Hq} Hkv={Hkv} L={L} D={D} bs={bs} causal={causal} density={density}", flush=True)
    nb = -(-L // 64) * 64 // bs
    rng = np.random.default_rng(L)
    pat = rng.random((1 if Hkv != Hq else Hq, nb, nb)) < density
    pat |= np.eye(nb, dtype=bool)[None]
    if causal:
        pat = np.tril(pat)
    if long_rows:
        pat[:, :64 // bs] = True
    sm = 1 / math.sqrt(D)
    q, k, v, do = make_qkv(B, L, L, Hq, Hkv, D, dtype, with_do=True)
    qo, ko, vo = (x.float().requires_grad_() for x in (q, k, v))
    ro, rl = oracle_fwd(qo, ko, vo, np.repeat(pat, Hq // pat.shape[0], axis=0), bs, sm, causal=causal)
    ro.backward(do.float())
    mod = SparseAttention(bs, torch.from_numpy(pat.astype(np.uint8)), causal=causal).to("cuda")
    qd, kd, vd = (x.cuda().requires_grad_() for x in (q, k, v))
    out, lse = mod(qd, kd, vd, sm, return_lse=True)
    out.backward(do.cuda())
    assert_close("O", out, ro, **TOL)
    assert_close("LSE", lse, rl, atol=LSE_TOL, rtol=0)
    assert_close("dQ", qd.grad, qo.grad, **TOL)
    assert_close("dK", kd.grad, ko.grad, **TOL)
    assert_close("dV", vd.grad, vo.grad, **TOL)


# (256 dims and zero-padded 128 dims multiply every quadrant of a step, the others only those with an attended block)
@pytest.mark.parametrize("D,bs,dtype,walk", [
    (256, 32, torch.bfloat16, False), (256, 16, torch.float16, True), (112, 32, torch.bfloat16, False), (112, 32, torch.float16, True),
    (128, 16, torch.bfloat16, False), (96, 32, torch.bfloat16, True), (64, 16, torch.float16, False), (64, 32, torch.bfloat16, True)])
def test_listed_tiles_without_an_attended_block(D, bs, dtype, walk, monkeypatch):
    """Entries of an empty mask in the column table add nothing, at any place of a column, as a column's only ones and where
    one head's entries follow another's: rows that a column meets in such a tile alone may hold anything."""
    print(f"case D={D} bs={bs} {dtype} walk={walk}", flush=True)
    Hq, Hkv, L, n, f = 4, 2, 256, 4, 64 // bs
    rng = np.random.default_rng(5)
    pat = np.tril(rng.random((Hq, n * f, n * f)) < 0.4) | np.eye(n * f, dtype=bool)[None]
    pat[:, 3 * f:, :3 * f] = False  # the last 64 queries attend their own tile only
    mod = SparseAttention(bs, torch.from_numpy(pat.astype(np.uint8))).to("cuda")
    ptr, entries = mod.masked_csc_ccol.cpu(), mod.masked_csc_row.cpu()
    columns = [[entries[h, ptr[h, c]:ptr[h, c + 1]].tolist() for c in range(n)] for h in range(Hq)]
    columns[1][2] = columns[2][0] = columns[3][1] = []

    def with_tables(cols):
        lens = torch.tensor([[len(c) for c in head] for head in cols])
        rows = torch.zeros(Hq, int(lens.sum(1).max()), 2, dtype=torch.int32)
        for h, head in enumerate(cols):
            flat = [e for c in head for e in c]
            rows[h, :len(flat)] = torch.tensor(flat, dtype=torch.int32)
        monkeypatch.setitem(mod._buffers, "masked_csc_ccol", torch.nn.functional.pad(lens.cumsum(1), (1, 0)).to(torch.int32).cuda())
        monkeypatch.setitem(mod._buffers, "masked_csc_row", rows.cuda())

    q, k, v, do = (x.cuda() for x in make_qkv(1, L, L, Hq, Hkv, D, dtype, with_do=True))
    q[:, 192:], v[:, 192:], do[:, 192:] = math.inf, -math.inf, math.inf

    def grads():
        xs = [x.clone().requires_grad_() for x in (q, k, v)]
        mod(*xs, 0.1).backward(do)
        ran = ops.last_bwd_kernels.decode()
        assert "mfma_dkdv_kernel" in ran and "SUB = true" in ran and ("per q head" in ran) != walk, ran
        return [x.grad[:, :192] for x in xs]

    monkeypatch.setitem(mod.kwargs, "row_lengths", ())
    monkeypatch.setattr(ops, "_bwd_workspace", not walk)
    with_tables(columns)
    want = grads()
    mixed = [[list(c) for c in head] for head in columns]
    for head in mixed:
        for c in head[:3]:
            for _ in range(int(rng.integers(0, 3)) + (not c)):
                c.insert(int(rng.integers(0, len(c) + 1)), [3, 0])
    with_tables(mixed)
    got = grads()
    for name, a, b in zip(("dQ", "dK", "dV"), got, want):
        assert torch.isfinite(b).all() and torch.equal(a, b), name
