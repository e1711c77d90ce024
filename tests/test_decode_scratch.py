"""Scratch of the split-KV decode kernels (no GPU needed: the query looks at sizes only).  A call of
dk_fwd_noalloc is refused when it needs more than the library's fixed scratch, so the need must not
grow for calls that fitted: it is compared with one fp32 partial per wave and at least two blocks."""
from __future__ import annotations

import ctypes as C

import pytest

from dkernel_amd import _lib


def _need(batch, ratio, dim, entries):
    """dk_fwd_workspace_bytes of a decode step: `batch` sequences, one kv head, rows of `entries` blocks."""
    a = _lib.FwdArgs()
    fake = 1 << 20  # never looked at
    for name, heads in (("q", ratio), ("k", 1), ("v", 1), ("o", ratio)):
        setattr(a, name, _lib.Tensor(fake, heads * dim * 64 * entries, dim, heads * dim))
    a.csr = _lib.Lut(fake, fake, 0, 0, 1, 1, entries, 64, 64, 1, entries, 0)
    a.seqs = _lib.Seqs(batch, 1, 64 * entries, 0, None, None, None, None)
    a.num_q_heads, a.num_kv_heads, a.head_dim = ratio, 1, dim
    a.dtype, a.causal, a.impl, a.sm_scale = _lib.DK_BF16, 1, _lib.DK_IMPL_AUTO, 0.1
    return _lib.lib().dk_fwd_workspace_bytes(C.byref(a))


def _cdiv(a, b):
    return -(-a // b)


def _partial_per_unit(batch, ratio, dim, entries):
    blocks = min(16, max(2, _cdiv(entries, max(4, _cdiv(1024, batch)))))
    units = max(_cdiv(entries, blocks), min(entries, 4))
    units = _cdiv(units, 4) * 4 if units > 4 else units
    return batch * ratio * units * (dim + 2) * 4


@pytest.mark.parametrize("dim", [64, 128, 256])
def test_calls_that_fitted_the_fixed_scratch_still_do(dim):
    limit, fitted = _lib.DK_NOALLOC_SCRATCH_BYTES, 0
    for entries in list(range(1, 41)) + [100, 128, 500, 1024]:
        for ratio in (1, 3, 8) if dim == 256 else (1, 3, 8, 32):  # (q of 32 heads beside 256-wide tiles: too much LDS)
            for batch in list(range(1, 64)) + list(range(64, 1100, 7)) + [2048, 4096]:
                if _partial_per_unit(batch, ratio, dim, entries) <= limit:
                    fitted += 1
                    need = _need(batch, ratio, dim, entries)
                    assert 0 < need <= limit, (batch, ratio, dim, entries, need)
    assert fitted > 1000


def test_rows_of_one_workgroup_need_one_place():
    assert _need(64, 32, 128, 1) == 64 * 32 * 130 * 4
    assert _need(1, 4, 128, 16) == 4 * (8 + 1) * 130 * 4  # eight workgroups of four half blocks, one slot
