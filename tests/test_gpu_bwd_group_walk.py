"""dK / dV passes whose workgroups walk a column for all q heads of a kv head: as one stream of steps against the oracle,
and cut into segments, as larger launches are, against the pass by q heads."""
import math

import numpy as np
import pytest
import torch

from dkernel_amd import LocalStrideSparseAttention, SparseAttention, ops
from helpers import F32_TOL, TOL, assert_close, make_qkv, oracle_fwd
from oracle import layout as OL

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _run(mod, q, k, v, do, sm):
    qd, kd, vd = (x.detach().to(DEV).requires_grad_() for x in (q, k, v))
    mod(qd, kd, vd, sm).backward(do.to(DEV))
    return [qd.grad, kd.grad, vd.grad], ops.last_bwd_kernels.decode()


# without a workspace every launch walks whole groups; fp32 with up to 64 head dims always does
@pytest.mark.parametrize("B,Hq,Hkv,L,Lk,D,bs,dtype,own_tables", [
    (1, 4, 2, 200, 200, 128, 64, torch.bfloat16, False),
    (2, 6, 2, 333, 333, 64, 64, torch.float16, False),
    (1, 4, 1, 250, 400, 96, 64, torch.bfloat16, False),   # keys before the queries
    (1, 4, 2, 300, 300, 128, 64, torch.bfloat16, True),   # every q head has a table of its own, some columns empty
    (1, 4, 2, 320, 320, 64, 16, torch.bfloat16, True),
    (1, 8, 2, 300, 300, 128, 32, torch.bfloat16, False),
    (1, 4, 2, 300, 300, 192, 64, torch.bfloat16, False),
    (1, 4, 2, 300, 300, 64, 64, torch.float32, True),
    (1, 4, 2, 300, 300, 80, 64, torch.float32, False)])
def test_stream_of_heads(B, Hq, Hkv, L, Lk, D, bs, dtype, own_tables, monkeypatch):
    print(f"case B={B} Hq={Hq} Hkv={Hkv} L={L} Lk={Lk} D={D} bs={bs} {dtype} own_tables={own_tables}", flush=True)
    sm = 1 / math.sqrt(D)
    n = -(-Lk // bs)
    if own_tables:
        rng = np.random.default_rng(3)
        bm = rng.random((Hq, n, n)) < 0.3
        bm[1, :, 1] = bm[2, :, 0] = False  # a head without entries in a column, between or before others
        bm &= np.tril(np.ones((n, n), dtype=bool))[None]
        bm[:, np.arange(2, n), np.arange(2, n)] = True
        bm[:, :2, 0] = True
        mod = SparseAttention(bs, torch.from_numpy(bm)).to(DEV)
    else:
        bm = OL.block_mask(Hq, n * bs, bs, 2, 3, num_kv_heads=Hkv)
        mod = LocalStrideSparseAttention(Hq, n * bs, bs, 2, 3, num_kv_heads=Hkv).to(DEV)
    q, k, v, do = make_qkv(B, L, Lk, Hq, Hkv, D, dtype, with_do=True)
    monkeypatch.setattr(ops, "_bwd_workspace", False)
    got, ran = _run(mod, q, k, v, do, sm)
    assert "per q head" not in ran and "group_sum" not in ran and "generic" not in ran, ran
    qo, ko, vo = (x.clone().float().requires_grad_() for x in (q, k, v))
    ro, _ = oracle_fwd(qo, ko, vo, bm, bs, sm, causal=True)
    ro.backward(do.float())
    for name, a, want in zip(("dQ", "dK", "dV"), got, (qo.grad, ko.grad, vo.grad)):
        assert_close(name, a, want, **(F32_TOL if dtype == torch.float32 else TOL))


# launches from some hundred steps per resident workgroup on (fp32 up to 64 dims: any size)
@pytest.mark.parametrize("B,Hq,Hkv,L,table,D,bs,dtype,cut", [
    (2, 32, 8, 4000, 4000, 128, 64, torch.bfloat16, True),
    (4, 32, 8, 2048, 3000, 128, 64, torch.float16, False),   # longest column below the average; a table for longer sequences
    (1, 32, 8, 6007, 7000, 96, 64, torch.bfloat16, True),
    (3, 24, 8, 4001, 4001, 64, 64, torch.bfloat16, True),
    (1, 32, 8, 3600, 3600, 160, 64, torch.bfloat16, True),
    (2, 32, 8, 4000, 4000, 128, 32, torch.bfloat16, True),
    (2, 4, 2, 1400, 2000, 64, 64, torch.float32, True),
    (1, 8, 2, 1401, 1401, 48, 64, torch.float32, True)])
def test_segments_of_groups(B, Hq, Hkv, L, table, D, bs, dtype, cut, monkeypatch):
    print(f"case B={B} Hq={Hq} Hkv={Hkv} L={L} table={table} D={D} bs={bs} {dtype}", flush=True)
    mod = LocalStrideSparseAttention(Hq, table, bs, 16 * 64 // bs, 8, num_kv_heads=Hkv).to(DEV)
    g = torch.Generator(device=DEV).manual_seed(1)
    q, k, v, do = (torch.randn(B, L, h, D, generator=g, device=DEV).to(dtype) for h in (Hq, Hkv, Hkv, Hq))
    got, ran = _run(mod, q, k, v, do, D ** -0.5)
    assert "per q head" not in ran and "group_sum" not in ran and ran.count("segment_sum_kernel") >= int(cut), ran
    monkeypatch.setitem(mod.kwargs, "row_lengths", ())
    whole, ran = _run(mod, q, k, v, do, D ** -0.5)
    assert "segment_sum_kernel" not in ran and ("group_sum" in ran or dtype == torch.float32), ran
    # (each side rounds its fp32 sums once: an ulp of the type apart; the sums themselves in fp32)
    ulp = {torch.float32: 2e-5, torch.float16: 1e-3, torch.bfloat16: 8e-3}[dtype]
    for name, a, b in zip(("dQ", "dK", "dV"), got, whole):
        assert_close(name, a, b, atol=ulp * float(b.float().abs().max()) / 8, rtol=ulp)


@pytest.mark.parametrize("B,Hq,Hkv,L,table,bs,walks", [
    (1, 32, 8, 1000, 8192, 64, False), (1, 32, 8, 2048, 32768, 64, False), (2, 24, 8, 700, 4096, 32, False),
    (4, 32, 8, 2048, 8192, 64, True)])
def test_short_call_of_a_module_for_long_sequences(B, Hq, Hkv, L, table, bs, walks):
    """The launches are planned by the call: the kernels, and (nothing being cut) the bits, of a module for that length."""
    g = torch.Generator(device=DEV).manual_seed(2)
    q, k, v, do = (torch.randn(B, L, h, 128, generator=g, device=DEV).to(torch.bfloat16) for h in (Hq, Hkv, Hkv, Hq))
    (got, ran), (want, ran_tight) = (
        _run(LocalStrideSparseAttention(Hq, n, bs, 16 * 64 // bs, 8, num_kv_heads=Hkv).to(DEV), q, k, v, do, 0.1) for n in (table, L))
    assert ran == ran_tight and ("per q head" not in ran) == walks, (ran, ran_tight)
    for name, a, b in zip(("dQ", "dK", "dV"), got, want):
        if "segment_sum" in ran:
            assert_close(name, a, b, atol=1e-3 * float(b.float().abs().max()), rtol=8e-3)
        else:
            assert torch.equal(a, b), name


def _check_against_oracle(mod, bm, bs, D, dtype, heads, lengths):
    sm = 1 / math.sqrt(D)
    for L, Lk in lengths:
        print(f"case D={D} bs={bs} {dtype} L={L} Lk={Lk}", flush=True)
        q, k, v, do = make_qkv(1, L, Lk, *heads, D, dtype, with_do=True)
        got, ran = _run(mod, q, k, v, do, sm)
        assert "mfma_dkdv" in ran and ("SUB = true" in ran) == (bs < 64) and "per q head" not in ran, ran
        qo, ko, vo = (x.clone().float().requires_grad_() for x in (q, k, v))
        ro, _ = oracle_fwd(qo, ko, vo, bm, bs, sm, causal=True)
        ro.backward(do.float())
        for name, a, want in zip(("dQ", "dK", "dV"), got, (qo.grad, ko.grad, vo.grad)):
            assert_close(f"{name} L={L} Lk={Lk}", a, want, **TOL)


SHORT = [(128, 64, torch.bfloat16), (64, 64, torch.float16), (256, 64, torch.bfloat16), (128, 32, torch.bfloat16), (64, 16, torch.float16),
         (256, 32, torch.bfloat16), (112, 32, torch.float16)]  # (the last two: masked steps of which no wave sits one out)


@pytest.mark.parametrize("D,bs,dtype", SHORT)
def test_short_columns(D, bs, dtype):
    """dK / dV of columns with one to five listed blocks (and of the call's part of them), fewer than the steps that are
    requested ahead and around the lengths of the rings, their last step whole, one row or one row short; the second head lists nothing
    below the diagonal."""
    n = 10 * 64 // bs
    bm = np.zeros((2, n, n), dtype=bool)
    for c in range(n):
        bm[0, c:c + 1 + c % 5, c] = True
    bm[1] = np.eye(n, dtype=bool)
    tiles = bm[0, :, :5].sum(0)
    assert list(tiles) == [1, 2, 3, 4, 5]
    mod = SparseAttention(bs, torch.from_numpy(bm)).to(DEV)
    _check_against_oracle(mod, bm, bs, D, dtype, (2, 2), (
        (1, 1), (31, 31), (32, 32), (33, 33), (65, 65), (97, 97), (320, 320), (353, 353), (384, 384), (609, 609), (640, 640), (40, 300)))


@pytest.mark.parametrize("D,bs,dtype", SHORT)
def test_short_columns_of_a_group(D, bs, dtype, monkeypatch):
    """The same where a workgroup goes on from head to head: columns in which the two heads of a group list none, one or two tiles
    each, in every combination, so that the stream ends, or changes heads, within the steps that
    are requested ahead."""
    n, first = 6, (0, 1, 2, 1, 0, 0)  # tiles; what head h lists in column 0
    tiles = np.zeros((6, n, n), dtype=bool)
    for h in range(6):
        for c in range(n):
            tiles[h, c:c + (c + first[h]) % 3, c] = True
        tiles[h, 0, 0] = True  # (every row has a key)
    lists = tiles.sum(1)
    pairs = {(int(a), int(b)) for h in (0, 2, 4) for a, b in zip(lists[h, 1:-1], lists[h + 1, 1:-1])}
    assert pairs == {(0, 1), (1, 2), (2, 0), (2, 1), (0, 2), (1, 0), (0, 0), (1, 1), (2, 2)}
    bm = np.kron(tiles, np.ones((1, 64 // bs, 64 // bs), dtype=bool))
    mod = SparseAttention(bs, torch.from_numpy(bm)).to(DEV)
    monkeypatch.setattr(ops, "_bwd_workspace", False)
    _check_against_oracle(mod, bm, bs, D, dtype, (6, 3), ((33, 33), (321, 321), (353, 353), (384, 384), (100, 350)))
