"""Split-operand products (fp32 operands in three bf16 parts, six products) on
the MI355X: through aar_gemm_f32 at shapes that the planner gives to them (which
the tests ask it), and every tile configuration by itself: whole tiles, remainders
in every extent, contractions shorter than and not a multiple of a K tile, K
splits, unaligned operands.

Tolerance: the matrix unit rounds once per 16 products, so an output's error is
a random walk of K / 16 roundings of at most 2^-24 of a partial sum, plus the
final rounding and the products left out (2^-25 each): normwise
2^-24 (2 + sqrt(K / 16)) against fp64.

Magnitudes the split does not cover (bf16 underflow and overflow, infinities,
NaN) go to the fp32 instruction: the same outputs are non-finite as in fp64
arithmetic and the others as precise."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

from devutil import Abi, split_plan

pytestmark = pytest.mark.gpu
NN, NT, TN = 0, 1, 2
f32, f64 = np.float32, np.float64


def _product(op, a, b, offset=0):
    """aar_gemm_f32, which must take the split-operand kernels."""
    abi = Abi()
    try:
        M = a.shape[1] if op == TN else a.shape[0]
        K = a.shape[0] if op == TN else a.shape[1]
        N = b.shape[0] if op == NT else b.shape[1]
        pa, pb, pc = abi.put(a, offset), abi.put(b, offset), abi.empty(M * N)
        wsb = abi.L.aar_gemm_f32_workspace_bytes(op, M, N, K)
        assert split_plan(abi.L, op, M, N, K, pa, pb), "this product runs on the fp32 instruction"
        abi.check(abi.L.aar_gemm_f32(op, M, N, K, pa, pb, pc, abi.alloc(wsb) if wsb else None, wsb, None))
        return abi.get(pc, (M, N))
    finally:
        abi.free()


def _exact(op, a, b):
    a, b = a.astype(f64), b.astype(f64)
    return (a.T if op == TN else a) @ (b.T if op == NT else b)


def _operands(op, M, N, K, seed):
    rng = np.random.default_rng(seed)
    a = rng.standard_normal((K, M) if op == TN else (M, K)).astype(f32)
    b = rng.standard_normal((N, K) if op == NT else (K, N)).astype(f32)
    return a, b


def _bound(K):
    return 2.0 ** -24 * (2 + np.sqrt(K / 16))


# every tile configuration is planned by one of them (aligned or off by one float)
SHAPES = [
    (2048, 1536, 600),   # 64 x 64 tiles
    (4095, 1537, 130),   # 256 x 128, a remainder of one in each extent
    (3000, 1153, 257),   # 128 x 128, a ragged K of one element
    (8192, 512, 1024),   # 128 x 64
    (4095, 4097, 65),    # a short contraction: two whole K tiles and a ragged one
    (1025, 771, 5001),   # K splits, the last one ragged
    (384, 384, 16384),   # a weight gradient: 128 x 192 tiles (unaligned 64 x 128), many splits
    (70, 70, 9000),      # one tile, many splits
]
@pytest.mark.parametrize("op", [NN, NT, TN])
@pytest.mark.parametrize("shape", SHAPES)
def test_split_product_against_fp64(gpu, op, shape):
    M, N, K = shape
    a, b = _operands(op, M, N, K, seed=M + N + K + op)
    for offset in (0, 1):  # 16-byte aligned operands, then off by one float
        c = _product(op, a, b, offset)
        r = _exact(op, a, b)
        assert np.linalg.norm(c - r) <= _bound(K) * np.linalg.norm(r), (op, shape, offset)
        assert np.array_equal(c, _product(op, a, b, offset))  # deterministic


@pytest.mark.parametrize("op", [NN, NT, TN])
@pytest.mark.parametrize("shape", [(2049, 1030, 130), (1025, 771, 5001)])
def test_split_product_magnitudes(gpu, op, shape):
    """Rows of A and columns of B from 1e-37 to 1e30, and elements of one row
    from 1e-40 to 1: every row of the result is as precise as its own scale."""
    M, N, K = shape
    a, b = _operands(op, M, N, K, seed=7)
    A, B = (a.T if op == TN else a), (b.T if op == NT else b)  # [M, K], [K, N] views
    for r, s in ((0, 1e-37), (1, 1e-30), (2, 1e-20), (3, 1e30), (M - 1, 1e-36)):
        A[r] *= f32(s)
    A[5] *= (10.0 ** -np.linspace(0, 40, K)).astype(f32)
    B[:, 1] *= f32(1e-25)
    A[6], B[:, 2] = 0.0, 0.0
    with np.errstate(over="ignore", under="ignore"):
        c, r = _product(op, a, b), _exact(op, a, b)
    for i in (0, 1, 2, 3, 5, 6, M - 1):
        keep = np.arange(N) != 1
        err, ref = np.linalg.norm(c[i, keep] - r[i, keep]), np.linalg.norm(r[i, keep])
        # (a scale of 1e-37 leaves subnormal operands and results, of 2^-149 steps)
        assert err <= 2 * _bound(K) * ref + 2.0 ** -149 * (np.sqrt(N) + K), i
    assert np.linalg.norm(c[10:, 1] - r[10:, 1]) <= 2 * _bound(K) * np.linalg.norm(r[10:, 1])
    assert not c[6].any() and not c[:, 2].any()


@pytest.mark.parametrize("op", [NN, NT, TN])
def test_split_product_non_finite(gpu, op):
    M, N, K = 2049, 1030, 130
    a, b = _operands(op, M, N, K, seed=9)
    A, B = (a.T if op == TN else a), (b.T if op == NT else b)
    A[3, 5], A[700, 0], A[M - 1, K - 1] = np.inf, np.nan, -np.inf
    B[7, 11], B[100, N - 1] = -np.inf, np.nan
    A[40, 9] = np.finfo(f32).max  # rounds to infinity in bf16, finite in fp32
    B[9, :] *= f32(1e-3)
    A[41], B[:, 20] = f32(3e38), f32(3e38)  # overflows to infinity
    with np.errstate(all="ignore"):
        c, r = _product(op, a, b), _exact(op, a, b).astype(f32)
    # (a sum of 3e38 terms of both signs leaves fp32's range on the way, to
    # either infinity and from there to NaN)
    ok = np.ones((M, N), bool)
    ok[41], ok[:, 20] = False, False
    assert np.array_equal(np.isnan(c) & ok, np.isnan(r) & ok)
    assert np.array_equal(np.isinf(c) & ok, np.isinf(r) & ok) and np.array_equal(np.sign(c[np.isinf(r) & ok]),
                                                                                np.sign(r[np.isinf(r) & ok]))
    assert c[41, 20] == np.inf
    good = np.isfinite(r) & ok
    good[40] = False
    assert np.linalg.norm((c - r)[good]) <= 2 * _bound(K) * np.linalg.norm(r[good])
    row = np.isfinite(r[40]) & ok[40]
    assert np.linalg.norm((c - r)[40, row]) <= 2 * _bound(K) * np.linalg.norm(r[40, row].astype(f64))


@pytest.mark.parametrize("op", [NN, NT, TN])
@pytest.mark.parametrize("shape", [(4095, 1537, 130), (2049, 1030, 257), (1025, 771, 5001)])
@pytest.mark.parametrize("scale", [0, 50, -60])
def test_split_product_selects_tiny_elements(gpu, op, shape, scale):
    """Every output is one element of A times a power of two, the elements of a
    row lying between fp32's smallest subnormal and 1e15: nothing else adds up,
    so each output is that element's exact product, whatever stands beside it.
    (At 2^-60 the small ones' products are rounded to subnormals: within one
    step of 2^-149 per part that is summed.)"""
    M, N, K = shape
    rng = np.random.default_rng(M + scale)
    x = (rng.uniform(1, 2, (M, K)) * 2.0 ** rng.uniform(-150, 50, (M, K)) * rng.choice([-1, 1], (M, K))).astype(f32)
    x[:, rng.integers(0, K, K // 8)] = 0.0
    x[::3, 1] = f32(1.0)
    rows = np.arange(N) % K
    sel = np.zeros((K, N), f32)
    sel[rows, np.arange(N)] = f32(2.0 ** scale)
    a = np.ascontiguousarray(x.T) if op == TN else x
    b = np.ascontiguousarray(sel.T) if op == NT else sel
    c, want = _product(op, a, b), x.astype(f64)[:, rows] * 2.0 ** scale
    if scale >= 0:
        np.testing.assert_array_equal(c, want)  # (products of a power of two are exact)
    else:
        assert (np.abs(c - want) <= 6 * 2.0 ** -149).all()
        big = np.abs(want) >= 2.0 ** -125  # the parts' products end at 2^-149 or above
        np.testing.assert_array_equal(c[big], want[big])


def test_split_product_tiny_beside_dense(gpu):
    """Tiny and subnormal elements beside ordinary ones in dense operands, zero
    rows and columns among them: the outputs feel none of it and stay as
    precise as without."""
    M, N, K = 2049, 1030, 257
    a, b = _operands(NN, M, N, K, seed=11)
    rng = np.random.default_rng(11)
    a[rng.random((M, K)) < 0.2] *= f32(1e-36)
    b[rng.random((K, N)) < 0.2] *= f32(1e-40)
    a[100:110], b[:, 70:75] = 0.0, 0.0
    c, r = _product(NN, a, b), _exact(NN, a, b)
    assert np.linalg.norm(c - r) <= _bound(K) * np.linalg.norm(r)
    assert not c[100:110].any() and not c[:, 70:75].any()


def _configs(L):
    out, tile = [], [ctypes.c_int() for _ in range(3)]
    while L.aar_gemm_f32_split_tile_config(len(out), *map(ctypes.byref, tile)) == 0:
        out.append(tuple(t.value for t in tile))
    return out


def test_planned_shapes_cover_the_configurations(gpu):
    L = Abi().L
    plans = [split_plan(L, op, *shape, addr, addr) for op in (NN, NT, TN) for shape in SHAPES for addr in (16, 20)]
    assert {p[0] for p in plans} == set(range(len(_configs(L))))
    assert any(p[1] > 1 for p in plans) and any(p[1] == 1 for p in plans)


@pytest.mark.parametrize("op", [NN, NT, TN])
@pytest.mark.parametrize("config", range(6))
def test_every_configuration(gpu, op, config):
    """Edges of the tiles and of the contraction: K below, at and past one and
    several K tiles (a ragged tile only, whole tiles only, both), chunks of K whose
    last one is shorter than a K tile, aligned operands and operands off by one."""
    abi = Abi()
    try:
        tiles = _configs(abi.L)
        assert len(tiles) == 6
        bm, bn, bk = tiles[config]
        cases = [(bm + 1, bn + 1, K, 1) for K in (1, 7, bk - 1, bk, bk + 1, 2 * bk, 2 * bk + 1, 5 * bk - 1)]
        cases += [(3, 5, 2 * bk + 3, 1), (2 * bm, bn, 3 * bk, 1), (bm - 1, 3 * bn - 31, 4 * bk, 1)]
        cases += [(bm + 1, bn - 1, 64 * 3 + r, 4) for r in (1, bk - 1, bk, 64)] + [(bm, bn, 128, 2)]
        for M, N, K, splits in cases:
            a, b = _operands(op, M, N, K, seed=M + K)
            for offset in (0, 1):
                pa, pb, pc = abi.put(a, offset), abi.put(b, offset), abi.put(np.full((M, N), np.nan, f32))
                ws = 4 * splits * M * N if splits > 1 else 0
                abi.check(abi.L.aar_gemm_f32_with_split_config(op, M, N, K, pa, pb, pc, abi.alloc(ws) if ws else None,
                                                               ws, config, splits, None))
                c, r = abi.get(pc, (M, N)), _exact(op, a, b)
                assert np.linalg.norm(c - r) <= _bound(K) * np.linalg.norm(r), (M, N, K, splits, offset)
    finally:
        abi.free()


def test_forced_configuration_arguments(gpu):
    abi = Abi()
    try:
        L, n, p = abi.L, len(_configs(abi.L)), abi.alloc(64 * 64 * 4)
        run = L.aar_gemm_f32_with_split_config
        assert run(NN, 64, 64, 64, p, p, p, None, 0, n, 1, None) == -1
        assert run(NN, 64, 64, 64, p, p, p, None, 0, -1, 1, None) == -1
        assert run(NN, 64, 64, 64, p, p, p, None, 0, 0, 0, None) == -1
        assert run(NN, 64, 64, 256, p, p, p, None, 0, 0, 2, None) == -2  # no workspace
        assert run(NT, 1, 1, 1 << 22, p, p, p, None, 0, 0, 1, None) == -3  # 32-bit offsets within a tile
    finally:
        abi.free()
