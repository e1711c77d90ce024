"""Decode rows that are cut over several workgroups and merged by the one that arrives last: one to
many half blocks (32 keys), odd counts, more than eight workgroups (two merge passes), every tile
width, masked tiles, scratch that holds arbitrary bytes, repeated calls (bit-identical: who arrives
last must not matter) against the fp32 oracle at the 16-bit bar."""
import ctypes as C
import math

import pytest
import torch

from dkernel_amd import LocalStrideSparseAttention, _lib, ops
from helpers import LSE_TOL, TOL, assert_close
from oracle import attention as OA
from oracle import layout as OL

pytestmark = pytest.mark.gpu
DEV = "cuda"
New = LocalStrideSparseAttention.__wrapped__


@pytest.mark.parametrize("ctx,D,bs,local,vert,dtype", [
    (1, 128, 64, 4, 2, torch.bfloat16),
    (32, 64, 64, 4, 2, torch.float16),
    (33, 128, 64, 4, 2, torch.bfloat16),
    (130, 128, 64, 4, 2, torch.bfloat16),      # three blocks: six units
    (1000, 96, 64, 16, 8, torch.float16),
    (4090, 128, 64, 4, 2, torch.bfloat16),     # 36 entries: 18 workgroups
    (4096, 64, 32, 4, 2, torch.bfloat16),      # masked tiles
    (2100, 192, 64, 4, 2, torch.bfloat16),
])
def test_one_sequence_against_the_oracle(ctx, D, bs, local, vert, dtype):
    print(f"case ctx={ctx} D={D} bs={bs}", flush=True)
    Hq, Hkv, Lmax = 8, 2, 4096
    sm = 1 / math.sqrt(D)
    g = torch.Generator().manual_seed(ctx)
    q = torch.randn(1, 1, Hq, D, generator=g).to(dtype)
    k, v = (torch.randn(1, ctx, Hkv, D, generator=g).to(dtype) for _ in range(2))
    bm = OL.block_mask(Hq, Lmax, bs, local, vert, num_kv_heads=Hkv)
    mask = OA.sequence_token_mask(bm, bs, 1, ctx)
    ro, rl = OA.dense_attention(q, k, v, torch.from_numpy(mask), sm)
    mod = New(Hq, Lmax, bs, local, vert, num_kv_heads=Hkv).to(DEV)
    dev = [x.to(DEV) for x in (q, k, v)]
    first = mod(*dev, sm, return_lse=True)
    assert _lib.lib().dk_last_kernels().startswith(b"decode_partial_kernel")
    assert_close("O", first[0], ro, **TOL)
    assert_close("LSE", first[1], rl, atol=LSE_TOL, rtol=0)
    for _ in range(20):
        again = mod(*dev, sm, return_lse=True)
        assert torch.equal(again[0], first[0]) and torch.equal(again[1], first[1])


@pytest.mark.parametrize("Hq,Hkv", [(6, 2), (16, 1), (12, 1)])
def test_groups_that_are_no_power_of_two_or_large(Hq, Hkv):
    """3, 12 and 16 q heads per kv head: the module finds runs of any length, so these groups decode on
    the split-KV kernels (and may page their keys) too."""
    print(f"case Hq={Hq} Hkv={Hkv}", flush=True)
    B, ctx, D, Lmax = 2, 700, 128, 1024
    sm = 1 / math.sqrt(D)
    g = torch.Generator().manual_seed(Hq)
    q = torch.randn(B, 1, Hq, D, generator=g).to(torch.bfloat16)
    k, v = (torch.randn(B, ctx, Hkv, D, generator=g).to(torch.bfloat16) for _ in range(2))
    bm = OL.block_mask(Hq, Lmax, 64, 2, 4, num_kv_heads=Hkv)
    ro, _ = OA.dense_attention(q, k, v, torch.from_numpy(OA.sequence_token_mask(bm, 64, 1, ctx)), sm)
    mod = New(Hq, Lmax, 64, 2, 4, num_kv_heads=Hkv).to(DEV)
    assert mod.lut_group % (Hq // Hkv) == 0
    out = mod(q.to(DEV), k.to(DEV), v.to(DEV), sm)
    assert _lib.lib().dk_last_kernels().startswith(b"decode_partial_kernel")
    assert_close("O", out, ro, **TOL)


@pytest.mark.parametrize("fill", [0x00, 0xff, 0x7f])
def test_scratch_may_hold_anything(fill):
    B, Hq, Hkv, L, D = 2, 8, 2, 3000, 128
    g = torch.Generator(device=DEV).manual_seed(1)
    q = torch.randn(B, 1, Hq, D, generator=g, device=DEV).to(torch.bfloat16)
    k, v = (torch.randn(B, L, Hkv, D, generator=g, device=DEV).to(torch.bfloat16) for _ in range(2))
    mod = New(Hq, 4096, 64, 4, 2, num_kv_heads=Hkv).to(DEV)
    want = mod(q, k, v, 0.1)
    out = torch.empty_like(q)
    a = _lib.FwdArgs()
    a.q, a.k, a.v, a.o = (ops._tensor4(x, 2, 1) for x in (q, k, v, out))
    a.lse = ops._rowvec(None)
    a.csr = ops._lut((mod.layout_csr_crow, mod.layout_csr_col, 64, 64), q.device, mod.lut_group, mod.lut_max_row)
    a.seqs = _lib.Seqs(B, 1, L, 0, None, None, None, None)
    a.num_q_heads, a.num_kv_heads, a.head_dim = Hq, Hkv, D
    a.dtype, a.causal, a.impl, a.sm_scale, a.stream = _lib.DK_BF16, 1, _lib.DK_IMPL_AUTO, 0.1, ops._stream()
    lib = _lib.lib()
    need = lib.dk_fwd_workspace_bytes(C.byref(a))
    ws = torch.full((need,), fill, dtype=torch.uint8, device=DEV)
    a.workspace, a.workspace_bytes = ws.data_ptr(), need
    for _ in range(3):  # the same scratch again, as the last call left it
        out.fill_(float("nan"))
        _lib.check(lib.dk_fwd(C.byref(a)))
        torch.cuda.synchronize()
        assert torch.equal(out, want)
