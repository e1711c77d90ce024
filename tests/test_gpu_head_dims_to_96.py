"""16-bit head dims of 72 - 96 multiply 96 of the 128 dims their tiles are laid out for (six k-steps, three
32-dim tiles); 104 - 120 multiply all of them.  Forward and backward on both sides of that line, in every form of
the kernels: split launches, row pairs, head groups, masked tiles, the dK/dV pass with and without its scratch."""
import math

import numpy as np
import pytest
import torch

from dkernel_amd import LocalStrideSparseAttention, _lib, ops
from helpers import LSE_TOL, TOL, assert_close, make_qkv, oracle_fwd
from oracle import layout as OL

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [72, 88, 96, 104])
@pytest.mark.parametrize("B,Hq,Hkv,L,bs,fixed_walk,workspace", [
    (1, 3, 3, 97, 64, False, True),    # split along the keys
    (2, 3, 3, 333, 64, True, True),    # row pairs
    (1, 8, 2, 450, 64, True, True),    # four heads a workgroup, dK / dV by q heads
    (1, 4, 2, 257, 64, True, False),   # two heads a workgroup, dK / dV by kv heads
    (1, 2, 2, 385, 32, True, True),    # masked tiles, one row
    (1, 4, 1, 321, 16, True, True)])   # masked tiles, head groups
def test_forward_and_backward(D, B, Hq, Hkv, L, bs, fixed_walk, workspace, monkeypatch):
    print(f"case D={D} B={B} Hq={Hq} Hkv={Hkv} L={L} bs={bs}", flush=True)
    monkeypatch.setattr(ops, "_bwd_workspace", workspace)
    dtype, sm = (torch.float16 if D == 88 else torch.bfloat16), 1 / math.sqrt(D)
    bm = OL.block_mask(Hq, -(-L // bs) * bs, bs, 2, 3, num_kv_heads=Hkv)
    q, k, v, do = make_qkv(B, L, L, Hq, Hkv, D, dtype, with_do=True)
    qo, ko, vo = (x.clone().float().requires_grad_() for x in (q, k, v))
    ro, rlse = oracle_fwd(qo, ko, vo, bm, bs, sm)
    ro.backward(do.float())
    mod = LocalStrideSparseAttention(Hq, -(-L // bs) * bs, bs, 2, 3, num_kv_heads=Hkv, fixed_walk=fixed_walk).to("cuda")
    qd, kd, vd = (x.cuda().requires_grad_() for x in (q, k, v))
    out, lse = mod(qd, kd, vd, sm, return_lse=True)
    ran = _lib.lib().dk_last_kernels().decode()
    assert (", 96 dims" in ran) == (D <= 96), ran
    out.backward(do.cuda())
    assert (b", 96 dims" in ops.last_bwd_kernels) == (D <= 96), ops.last_bwd_kernels
    for name, got, want in (("O", out, ro), ("dQ", qd.grad, qo.grad), ("dK", kd.grad, ko.grad), ("dV", vd.grad, vo.grad)):
        assert_close(name, got, want, **TOL)
    assert_close("LSE", lse, rlse, atol=LSE_TOL, rtol=0)
    assert np.isfinite(ro.detach().numpy()).all()
