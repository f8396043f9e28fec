"""Fused and batched products that stay on the fp32 instruction: short contractions,
where the split-operand kernels gain nothing.  The same checks as in the files
the tests come from, at shapes whose plan is asked for first; the fused calls must
be taken."""
from __future__ import annotations

import pytest

import oracle as O
from devutil import Abi, split_plan
from test_colsum_gemm_gpu import test_colsum_gemm_matches_product_and_colsum as check_colsum
from test_extra_ops_gpu import test_bmm_one_tile_per_cu_grid as check_bmm
from test_linear_gpu import test_linear_bit_identical_to_composition as check_linear
from test_relu_bits_gpu import check_taken, test_bits_forward_and_masked_backward as check_bits
from test_residual_gpu import test_abi_gemm_add_epilogues as check_add

pytestmark = pytest.mark.gpu
NN, NT, TN = 0, 1, 2


def _on_fp32(op, M, N, K, batch=1):
    assert split_plan(Abi().L, op, M, N, K, batch=batch) is None


# (M, N, K): 128 x 128 and 64 x 64 tiles over three 64-row chunks, then each other
# tile without K groups that is planned for 64
@pytest.mark.parametrize("M,N,K", [(1024, 4096, 192), (512, 2304, 192), (3072, 3072, 64), (2304, 2304, 64),
                                   (1536, 4096, 64), (2048, 2048, 64)])
def test_column_sums(gpu, M, N, K):
    _on_fp32(TN, M, N, K)
    check_colsum(gpu, M, N, K, True)


# (M, H, d, N2) as in test_relu_bits_gpu: 32-row wave tiles with a 4-row last word,
# 64-row ones
@pytest.mark.parametrize("M,H,d,N2", [(4096, 1536, 64, 64), (4004, 1536, 96, 64), (16384, 1536, 32, 32),
                                      (16384, 1536, 32, 48)])
def test_relu_bits(gpu, M, H, d, N2):
    _on_fp32(NT, M, H, d)
    _on_fp32(NN, M, H, N2)
    check_taken(NT, M, H, d)
    check_taken(NN, M, H, N2)
    check_bits(gpu, M, H, d, N2)


@pytest.mark.parametrize("lead,K,N", [((372,), 64, 16384), ((480,), 64, 20000)])
def test_linear_bias(gpu, lead, K, N):
    _on_fp32(NT, lead[0], N, K)
    check_linear(gpu, lead, K, N)


@pytest.mark.parametrize("K", [64, 96])
def test_residual_adds(gpu, K):
    _on_fp32(NT, 16100, 384, K)  # the 8-wave 128 x 192 tile, a ragged last row tile
    check_add(gpu, 16100, 384, K, 0)


@pytest.mark.parametrize("op", O.BMM_OPS)
def test_batched(gpu, op):
    _on_fp32({"bmm": NN, "bmm_a_bt": NT, "bmm_at_b": TN}[op], 8192, 384, 64, batch=2)
    check_bmm(gpu, op, K=64)  # the 128 x 192 tiles, one per CU
