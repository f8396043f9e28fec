"""The GEMM planner without a device (its plans depend on the shape, the layout and
the operands' alignment): the workspace that a product asks for buys the plan that
it would have with any amount, and NN products of the shapes whose fp32 plan has the
mask-bits epilogue keep their K whole."""
from __future__ import annotations

import itertools

import pytest

from devutil import Abi, split_plan

NN, NT, TN = 0, 1, 2
ALIGNED, OFF_BY_ONE = 64, 68
UNLIMITED = 1 << 62


@pytest.mark.parametrize("op", [NN, NT, TN])
def test_queried_workspace_buys_the_unlimited_plan(op):
    L = Abi().L
    taken = 0
    for M, N, K in itertools.product((64, 100, 384, 1024, 1537, 4096, 16384), (65, 256, 384, 1025, 2304, 3072),
                                     (33, 64, 130, 384, 1025, 4096, 16384)):
        for addr in (ALIGNED, OFF_BY_ONE):
            plan = split_plan(L, op, M, N, K, addr, addr)
            assert plan == split_plan(L, op, M, N, K, addr, addr, ws=UNLIMITED), (M, N, K, addr)
            # (without scratch K stays whole)
            alone = split_plan(L, op, M, N, K, addr, addr, ws=0)
            assert alone is None or alone[1] == 1
            taken += plan is not None
    assert taken > 100


def test_masked_products_keep_k_whole():
    L = Abi().L
    for shape in [(2304, 2304, 1920), (2304, 2304, 2560), (1920, 6144, 3072), (3072, 1920, 16384)]:
        assert split_plan(L, NN, *shape)[1] == 1
        assert split_plan(L, TN, *shape)[1] > 1  # the same product without that epilogue


def test_plan_arguments():
    L = Abi().L
    for args in [(3, 1, 8, 8, 8), (0, 0, 8, 8, 8), (0, 1, 0, 8, 8), (0, 1, 8, 8, 0)]:
        assert L.aar_gemm_f32_split_plan(*args, None, None, 0, None, None) == -1
    assert L.aar_gemm_f32_split_tile_config(-1, None, None, None) == -1
