"""How a workgroup finds its sequence among packed ones: up to 64 sequences every wave scans their lengths,
one per lane; beyond, running counts are bisected.  At the edges of the two ways, with empty sequences at
the front, in the middle and at the end, through the row-pair, the head-group and the fp32 kernels."""
import math

import numpy as np
import pytest
import torch

from dkernel_amd import LocalStrideSparseAttention
from helpers import F32_TOL, LSE_TOL, TOL, assert_close
from oracle import attention as OA
from oracle import layout as OL

pytestmark = pytest.mark.gpu
New = LocalStrideSparseAttention.__wrapped__


@pytest.mark.parametrize("Hq,Hkv,dtype", [(8, 8, torch.bfloat16), (8, 2, torch.float16), (8, 4, torch.float32)])
@pytest.mark.parametrize("nseq", [1, 3, 63, 64, 65])
def test_every_token_gets_its_own_sequence(Hq, Hkv, dtype, nseq):
    print(f"case Hq={Hq} Hkv={Hkv} dtype={dtype} nseq={nseq}", flush=True)
    D, bs, longest = 64, 64, 3072
    rng = np.random.default_rng(nseq)
    lens = [int(x) for x in rng.integers(1, 150, nseq)]
    lens[nseq // 2] = 3000  # (more tiles than the kernel for small launches takes)
    if nseq > 2:
        lens[0] = lens[-1] = 0
    if nseq > 3:
        lens[5] = lens[6] = 0
    g = torch.Generator().manual_seed(20)
    q, k, v = (torch.randn(sum(lens), h, D, generator=g).to(dtype) for h in (Hq, Hkv, Hkv))
    cu = [0] + [int(x) for x in np.cumsum(lens)]
    sm = 1 / math.sqrt(D)
    mod = New(Hq, longest, bs, 2, 3, num_kv_heads=Hkv).to("cuda")
    bm = OL.block_mask(Hq, longest, bs, 2, 3, num_kv_heads=Hkv)
    out, lse = mod(q.cuda(), k.cuda(), v.cuda(), sm, cu_seqlen_k=torch.tensor(cu, dtype=torch.int32, device="cuda"),
                   return_lse=True)
    tol, lse_tol = (F32_TOL, 1e-4) if dtype == torch.float32 else (TOL, LSE_TOL)
    for i in sorted({0, 1, 4, 7, nseq // 2, nseq - 2, nseq - 1} & set(range(nseq))):
        s, e = cu[i], cu[i + 1]
        if e == s:
            continue
        mask = torch.from_numpy(OA.sequence_token_mask(bm, bs, e - s, e - s))
        ro, rl = OA.dense_attention(*(x[None, s:e].float() for x in (q, k, v)), mask, sm)
        assert_close(f"O[{i}]", out[s:e], ro[0], **tol)
        assert_close(f"LSE[{i}]", lse[:, s:e], rl[0], atol=lse_tol, rtol=0)
    assert torch.isfinite(out).all() and torch.isfinite(lse).all()
