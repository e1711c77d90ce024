"""fixed_walk=True: the prefill of a sequence gives the same bits alone, in padded and packed batches and
in batches of any size, although a launch of the sequence alone is small enough to be split along the keys
otherwise.  Every kernel of larger launches: head groups, row pairs, single rows, masked tiles, tile widths."""
import pytest
import torch

from dkernel_amd import LocalStrideSparseAttention, _lib
from helpers import make_qkv

pytestmark = pytest.mark.gpu
DEV = "cuda"
New = LocalStrideSparseAttention.__wrapped__


def _kernel():
    return _lib.lib().dk_last_kernels().decode()


@pytest.mark.parametrize("Hq,Hkv,D,bs,causal,dtype", [
    (8, 2, 128, 64, True, torch.bfloat16), (4, 4, 128, 64, True, torch.float16), (6, 3, 64, 128, False, torch.bfloat16),
    (4, 4, 128, 32, True, torch.bfloat16),  # (masked tiles: single rows alone, row pairs in the batch)
    (4, 4, 96, 16, True, torch.float16), (4, 2, 64, 32, False, torch.bfloat16), (2, 2, 192, 32, True, torch.bfloat16),
    (4, 2, 256, 64, True, torch.bfloat16)])
def test_prefill_does_not_depend_on_the_batch(Hq, Hkv, D, bs, causal, dtype):
    print(f"case Hq={Hq} Hkv={Hkv} D={D} bs={bs} causal={causal}", flush=True)
    L, lens = 512, [300, 512, 1, 130, 77]
    B, sm = len(lens), D ** -0.5
    q, k, v = (x.to(DEV) for x in make_qkv(B, L, L, Hq, Hkv, D, dtype))
    kw = dict(num_kv_heads=Hkv, causal=causal)
    mod = New(Hq, L, bs, 2, 3, fixed_walk=True, **kw).to(DEV)
    assert not mod.kwargs["unsorted_rows"]
    n = torch.tensor(lens, dtype=torch.int32, device=DEV)
    cu = torch.cat([torch.zeros_like(n[:1]), n.cumsum(0, dtype=torch.int32)])
    alone = []
    for b in range(B):
        row = [x[b:b + 1, :lens[b]].contiguous() for x in (q, k, v)]
        alone.append(mod(*row, sm, return_lse=True))
        assert "split" not in _kernel(), _kernel()
    New(Hq, L, bs, 2, 3, **kw).to(DEV)(*row, sm)
    assert "split" in _kernel(), _kernel()  # what the default runs
    packed = mod(*(torch.cat([x[b, :lens[b]] for b in range(B)]) for x in (q, k, v)), sm, cu_seqlen_k=cu, return_lse=True)
    right = mod(q, k, v, sm, seqlens=n, return_lse=True)
    left = mod(*(torch.stack([x[b].roll(L - lens[b], 0) for b in range(B)]) for x in (q, k, v)), sm, left_paddings=L - n,
               return_lse=True)
    many = mod(*(x.repeat(40, 1, 1, 1) for x in (q, k, v)), sm, seqlens=n.repeat(40), return_lse=True)
    for b in range(B):
        o, lse = alone[b][0][0], alone[b][1][0]
        i, m = int(cu[b]), lens[b]
        for got_o, got_lse in ((packed[0][i:i + m], packed[1][:, i:i + m]), (right[0][b, :m], right[1][b, :, :m]),
                               (left[0][b, L - m:], left[1][b, :, L - m:]), (many[0][b + 35 * B, :m], many[1][b + 35 * B, :, :m])):
            assert torch.equal(got_o, o) and torch.equal(got_lse, lse), b


def test_default_and_explicit_choice():
    assert New(2, 512, 64, 2, 3).kwargs["fixed_walk"] is False
    from dkernel_amd import SparseAttention
    pattern = torch.eye(16) + torch.eye(16).roll(1, 0)
    pattern[:2] = 1
    assert SparseAttention(64, pattern, causal=False).kwargs["fixed_walk"] is True
    assert SparseAttention(64, pattern, causal=False, fixed_walk=False).kwargs["fixed_walk"] is False
