"""The forward kernels of launches that do not fit the chip at once (mfma_fwd_kernel: head groups, row pairs,
single rows, plain and masked tiles, every tile width), at sizes that the dense oracle can afford.  Launches this
small are split along the keys by default and run another kernel; fixed_walk keeps them on the one of larger
launches.  First the parity, padding, packing, rotation and random tests of the other files again under it, then
masked tables in every form of the kernel, each named by dk_last_kernels()."""
import math

import numpy as np
import pytest
import torch

from dkernel_amd import LocalStrideSparseAttention, SparseAttention, _lib
from helpers import LSE_TOL, TOL, assert_close, make_qkv, oracle_fwd
from test_gpu_masked_quadrants import test_sparse_tiles  # noqa: F401
from test_gpu_merged_rows import test_merged_rows_that_widen_the_pattern  # noqa: F401
from test_gpu_packed_search import test_every_token_gets_its_own_sequence  # noqa: F401
from test_gpu_padding_rows import test_rows_without_queries_are_cleared  # noqa: F401
from test_gpu_parity import (  # noqa: F401
    test_c4_user_pattern_varlen_partitions, test_dims_dtypes_block_sizes, test_dims_not_power_of_two, test_gqa,
    test_grad_through_lse, test_head_dims_below_tile_width, test_kernel_tile_sizes_on_the_matrix_cores,
    test_keys_broadcast_along_tokens, test_large_blocks_run_on_split_tiles, test_left_padded_prefill, test_noncausal,
    test_packed_chunked_prefill_every_sequence_starts_inside_a_block, test_packed_prefill_with_hundreds_of_sequences,
    test_packed_varlen_prefill_and_decode, test_patterns, test_ragged_lengths, test_right_padded_prefill,
    test_row_pairs_user_pattern_and_offsets, test_seq_dim_and_non_contiguous, test_seq_partition_with_backward)
from test_gpu_random_configs import (  # noqa: F401
    test_random_config_matches_generic_kernels_and_oracle, test_random_inference_config_matches_generic_kernels_and_oracle,
    test_random_user_pattern_matches_generic_kernels_and_oracle)
from test_gpu_uneven_heads import (  # noqa: F401
    test_forward_and_backward_match_the_oracle, test_padded_and_packed_prefill_do_not_depend_on_the_rotation)

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def one_walk(monkeypatch):
    """Modules are constructed with fixed_walk=True (the local-stride class keeps its latest ones)."""
    init = SparseAttention.__init__
    monkeypatch.setattr(SparseAttention, "__init__", lambda self, *a, **kw: init(self, *a, **{"fixed_walk": True, **kw}))
    LocalStrideSparseAttention.cache_clear()
    yield
    LocalStrideSparseAttention.cache_clear()


@pytest.fixture
def impl():
    return "auto"


def test_small_launches_are_not_split():
    mod = LocalStrideSparseAttention(4, 256, 64, 2, 3).to("cuda")
    q, k, v = (x.cuda() for x in make_qkv(1, 256, 256, 4, 4, 128, torch.bfloat16))
    mod(q, k, v)
    assert _lib.lib().dk_last_kernels().startswith(b"mfma_fwd_kernel ")


# (128-wide row pairs: from 385 pairs of 128 tokens x one head on, 321 with padded head dims)
PAIRS, SINGLE, TWO, FOUR = "SUB = true]", "G = 1,", "G = 2,", "G = 4,"


@pytest.mark.parametrize("B,Hq,Hkv,L,D,form", [
    (1, 2, 2, 700, 64, PAIRS), (2, 3, 3, 330, 40, PAIRS), (4, 32, 32, 400, 128, PAIRS), (4, 28, 28, 300, 96, PAIRS),
    (1, 2, 2, 450, 256, PAIRS), (1, 2, 2, 330, 200, PAIRS),
    (1, 2, 2, 700, 128, SINGLE), (2, 2, 2, 333, 104, SINGLE),
    (1, 4, 2, 513, 128, TWO), (1, 6, 3, 260, 80, TWO), (1, 8, 2, 450, 64, TWO), (2, 2, 1, 321, 24, TWO), (1, 4, 1, 400, 256, TWO),
    (1, 2, 1, 257, 136, TWO),
    (1, 8, 2, 513, 128, FOUR), (2, 4, 1, 300, 112, FOUR)])
@pytest.mark.parametrize("bs,causal,dtype", [(32, True, torch.bfloat16), (16, True, torch.float16), (32, False, torch.float16),
                                             (16, False, torch.bfloat16)])
def test_masked_tables(B, Hq, Hkv, L, D, form, bs, causal, dtype):
    """Sparse random blocks: most tiles hold one or two quadrants, rows of a pair share few columns."""
    print(f"case B={B} Hq={Hq} Hkv={Hkv} L={L} D={D} {form} bs={bs} causal={causal}", flush=True)
    nb = -(-L // 64) * 64 // bs
    rng = np.random.default_rng(L + D)
    pat = (rng.random((1 if Hkv != Hq else Hq, nb, nb)) < 2 / math.sqrt(nb) / (64 // bs)) | np.eye(nb, dtype=bool)[None]
    if causal:
        pat = np.tril(pat)
    sm = 1 / math.sqrt(D)
    q, k, v = make_qkv(B, L, L, Hq, Hkv, D, dtype)
    ro, rl = oracle_fwd(q.float(), k.float(), v.float(), np.repeat(pat, Hq // pat.shape[0], axis=0), bs, sm, causal=causal)
    mod = SparseAttention(bs, torch.from_numpy(pat.astype(np.uint8)), causal=causal).to("cuda")
    mod.kwargs["unsorted_rows"] = False  # (random rows can look like global ones, which run as single rows)
    out, lse = mod(q.cuda(), k.cuda(), v.cuda(), sm, return_lse=True)
    ran = _lib.lib().dk_last_kernels().decode()
    assert ran.startswith(("mfma_fwd_kernel ", "mfma_fwd_kernel, heads in rotation ")) and form in ran, ran
    assert_close("O", out, ro, **TOL)
    assert_close("LSE", lse, rl, atol=LSE_TOL, rtol=0)
