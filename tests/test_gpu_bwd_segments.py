"""Backward launches that cut long rows (dQ, with the table's own order) and long columns (dK / dV) into segments
of their own workgroups: against the oracle, and against the same call without the lengths that allow it (no more
than the rounding of another order of the sums apart)."""
import math

import numpy as np
import pytest
import torch

from dkernel_amd import LocalStrideSparseAttention, SparseAttention, ops
from helpers import F32_TOL, TOL, assert_close, make_qkv, oracle_fwd
from oracle import layout as OL

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _global_pattern(heads, n, block, causal, seed=5):
    rng = np.random.default_rng(seed)
    i = np.arange(n)
    pat = np.zeros((heads, n, n), dtype=bool)
    for h in range(heads):
        pat[h] = np.abs(i[:, None] - i[None, :]) <= 1 + h % 2
        g = (128 if h % 2 else 64) // block
        pat[h, :g, :] = True
        pat[h, :, :g] = True
        pat[h, n - 8 - h if causal else (3 * h + 9) % n, :] = True
        pat[h] |= rng.random((n, n)) < 1.5 / n
        if causal:
            pat[h] &= i[:, None] >= i[None, :]
            pat[h, i, i] = True
    return pat


def _run(mod, q, k, v, do, sm):
    qd, kd, vd = (x.to(DEV).requires_grad_() for x in (q, k, v))
    out = mod(qd, kd, vd, sm)
    out.backward(do.to(DEV))
    return [qd.grad, kd.grad, vd.grad], ops.last_bwd_kernels.decode()


def _check(mod, q, k, v, do, bm, bs, sm, causal, cut, monkeypatch):
    dtype = q.dtype
    qo, ko, vo = (x.clone().float().requires_grad_() for x in (q, k, v))
    ro, _ = oracle_fwd(qo, ko, vo, bm, bs, sm, causal=causal)
    ro.backward(do.float())
    got, ran = _run(mod, q, k, v, do, sm)
    assert ran.count("segment_sum_kernel") == cut, ran
    monkeypatch.setitem(mod.kwargs, "row_lengths", ())
    whole, ran = _run(mod, q, k, v, do, sm)
    assert "segment_sum_kernel" not in ran, ran
    tol = F32_TOL if dtype == torch.float32 else TOL
    # (each side rounds its fp32 sum once: an ulp of the type apart; the sums of a few hundred terms in fp32 themselves)
    ulp = {torch.float32: 2e-5, torch.float16: 1e-3, torch.bfloat16: 8e-3}[dtype]
    for name, a, b, want in zip(("dQ", "dK", "dV"), got, whole, (qo.grad, ko.grad, vo.grad)):
        assert_close(name, a, want, **tol)
        assert_close(name + " cut / whole", a, b, atol=ulp * float(b.float().abs().max()) / 8, rtol=ulp)


# columns: local window and vertical columns, few heads
@pytest.mark.parametrize("B,Hq,Hkv,L,Lk,table,D,bs,dtype", [
    (1, 2, 2, 1500, 1500, 1500, 128, 64, torch.bfloat16),
    (2, 4, 2, 1411, 1411, 1500, 64, 64, torch.float16),       # grouped heads: partials per q head, then their sum
    (1, 3, 3, 1400, 1500, 2500, 96, 64, torch.bfloat16),      # keys before the queries; a table for longer sequences
    (1, 4, 1, 1400, 1400, 3000, 128, 64, torch.bfloat16),
    (1, 2, 2, 1400, 1400, 1400, 192, 64, torch.bfloat16),     # 256-wide tile
    (1, 2, 2, 1400, 1400, 1400, 128, 32, torch.bfloat16),     # masked tiles
    (1, 2, 2, 1400, 1400, 2000, 104, 16, torch.float16),
    (1, 2, 2, 1400, 1400, 1400, 128, 128, torch.bfloat16),    # blocks split into tiles
    (1, 3, 3, 1500, 1500, 1500, 64, 64, torch.float32),
    (1, 2, 2, 1301, 1500, 2500, 100, 64, torch.float32),
    (2, 4, 2, 1400, 1400, 1400, 128, 64, torch.float32)])
def test_long_columns(B, Hq, Hkv, L, Lk, table, D, bs, dtype, monkeypatch):
    print(f"case B={B} Hq={Hq} Hkv={Hkv} L={L} Lk={Lk} D={D} bs={bs} {dtype}", flush=True)
    sm = 1 / math.sqrt(D)
    n = -(-Lk // bs)
    bm = OL.block_mask(Hq, n * bs, bs, max(1, 128 // bs), 3, num_kv_heads=Hkv)
    mod = LocalStrideSparseAttention(Hq, table, bs, max(1, 128 // bs), 3, num_kv_heads=Hkv).to(DEV)
    q, k, v, do = make_qkv(B, L, Lk, Hq, Hkv, D, dtype, with_do=True)
    _check(mod, q, k, v, do, bm, bs, sm, True, 1, monkeypatch)


# rows and columns: global blocks, heads of different lengths
@pytest.mark.parametrize("B,Hq,Hkv,L,D,bs,dtype,causal,cut", [
    (1, 3, 3, 1400, 64, 64, torch.bfloat16, False, 2),
    (2, 2, 2, 1390, 128, 64, torch.float16, False, 2),
    (1, 4, 2, 1400, 128, 64, torch.bfloat16, False, 2),
    (1, 2, 2, 1400, 80, 64, torch.bfloat16, False, 2),
    (1, 2, 2, 1400, 64, 32, torch.float16, False, 2),
    (1, 2, 2, 1420, 128, 32, torch.bfloat16, False, 2),
    (1, 2, 2, 1400, 160, 64, torch.bfloat16, False, 1),       # 256-wide tile: columns only
    (1, 2, 2, 2600, 128, 64, torch.bfloat16, True, 2),
    (1, 3, 3, 1400, 64, 64, torch.float32, False, 2),
    (1, 2, 2, 1400, 128, 64, torch.float32, False, 2)])
def test_global_rows_and_columns(B, Hq, Hkv, L, D, bs, dtype, causal, cut, monkeypatch):
    print(f"case B={B} Hq={Hq} Hkv={Hkv} L={L} D={D} bs={bs} {dtype} causal={causal}", flush=True)
    sm = 1 / math.sqrt(D)
    pat = _global_pattern(Hkv, -(-L // bs), bs, causal)
    mod = SparseAttention(bs, torch.from_numpy(pat), causal=causal).to(DEV)
    assert mod.kwargs["unsorted_rows"]
    q, k, v, do = make_qkv(B, L, L, Hq, Hkv, D, dtype, with_do=True)
    _check(mod, q, k, v, do, np.repeat(pat, Hq // Hkv, axis=0), bs, sm, causal, cut, monkeypatch)


def test_queries_that_start_inside_a_pair(monkeypatch):
    pat = _global_pattern(2, 44, 64, True)
    mod = SparseAttention(64, torch.from_numpy(pat), causal=True).to(DEV)
    q, k, v, do = make_qkv(1, 64 * 37 + 7, 64 * 44 - 20, 2, 2, 128, torch.bfloat16, with_do=True)
    _check(mod, q, k, v, do, pat, 64, 0.1, True, 2, monkeypatch)


def test_scratch_too_small_for_the_segments(monkeypatch):
    """The library takes what fits: without room for the partial sums no row is cut."""
    mod = LocalStrideSparseAttention(4, 1500, 64, 2, 3, num_kv_heads=2).to(DEV)
    q, k, v, do = make_qkv(1, 1500, 1500, 4, 2, 128, torch.bfloat16, with_do=True)
    got, ran = _run(mod, q, k, v, do, 0.1)
    assert "segment_sum_kernel" in ran and "per q head" in ran
    group = 2 * 4 * 1500 * 128 * 4
    ask = ops._lib.lib().dk_bwd_balanced_workspace_bytes

    class Lib:
        def __getattr__(self, name):
            return (lambda *a: min(ask(*a), group)) if name == "dk_bwd_balanced_workspace_bytes" else getattr(ops._lib.lib.__wrapped__(), name)
    real = ops._lib.lib
    fake = Lib()
    monkeypatch.setattr(ops._lib, "lib", lambda: fake)
    ops._lib.lib.__wrapped__ = real
    small, ran = _run(mod, q, k, v, do, 0.1)
    assert "segment_sum_kernel" not in ran and "per q head" in ran, ran
    for a, b in zip(got, small):
        assert_close("grad", a, b, atol=1e-3 * float(b.float().abs().max()), rtol=8e-3)


@pytest.mark.parametrize("Hq,Hkv,D,bs,dtype", [(2, 2, 128, 64, torch.bfloat16), (4, 2, 64, 64, torch.bfloat16),
                                               (2, 2, 64, 32, torch.bfloat16), (2, 2, 64, 64, torch.float32)])
def test_columns_in_any_order_without_lengths(Hq, Hkv, D, bs, dtype, monkeypatch):
    """dk_bwd without the lengths takes the entries of a column in any order, also of a table for longer sequences."""
    L, table = 700, 1500
    mod = LocalStrideSparseAttention(Hq, table, bs, 128 // bs, 3, num_kv_heads=Hkv).to(DEV)
    monkeypatch.setitem(mod.kwargs, "row_lengths", ())
    name = "masked_csc" if bs < 64 else "layout_csc"
    ptr, rows = getattr(mod, name + "_ccol").cpu(), getattr(mod, name + "_row")
    mixed = rows.cpu().clone()
    g = torch.Generator().manual_seed(1)
    for h in range(ptr.size(0)):
        for a, b in zip(ptr[h].tolist(), ptr[h].tolist()[1:]):
            mixed[h, a:b] = mixed[h, a:b][torch.randperm(b - a, generator=g)]
    q, k, v, do = make_qkv(1, L, L, Hq, Hkv, D, dtype, with_do=True)
    want, _ = _run(mod, q, k, v, do, 0.1)
    monkeypatch.setitem(mod._buffers, name + "_row", mixed.to(DEV))
    got, ran = _run(mod, q, k, v, do, 0.1)
    assert "generic" not in ran, ran
    tol = F32_TOL if dtype == torch.float32 else TOL
    for what, a, b in zip(("dQ", "dK", "dV"), got, want):
        assert_close(what, a, b, **tol)
