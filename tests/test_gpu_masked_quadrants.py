"""Masked 64 x 64 tiles (pattern blocks of 16 and 32): the kernels multiply 32 x 32 quadrants and leave out those
that hold no attended block.  Sparse random patterns, in which most tiles hold one or two quadrants and single
16-token blocks inside them, at every tile width, forward and backward, against the fp32 oracle at the 16-bit bar.
(The first six forwards are split along the keys, the others run single rows; row pairs and head groups:
test_gpu_large_launch_kernels.py.)"""
import math

import numpy as np
import pytest
import torch

from dkernel_amd import SparseAttention
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
