"""The forward on the bf16 matrix cores (operands in three bf16 parts) against
float64: head dims that fill and half fill the padded width,
sequences at the edges of tiles and blocks past the lengths that keep the fp32
instruction, and magnitudes that the split hands
to the fp32 instruction.  Bound on the relative 2-norm error of O and lse:
5e-6, the rounding of fp32 sums over d <= 64 products in S (at most about
sqrt(64) 2^-24 |S| ~ 2e-6 of P at |S| <= 4) and of O's over the keys (3e-7)."""
from __future__ import annotations

import ctypes
import math

import numpy as np
import pytest

from devutil import Abi

pytestmark = pytest.mark.gpu
f32 = np.float32


def _exact(q, k, v, causal):
    q, k, v = (t.astype(np.float64) for t in (q, k, v))
    T, d = q.shape[-2:]
    s = q @ k.swapaxes(-1, -2) / math.sqrt(d)
    if causal:
        s = np.where(np.triu(np.ones((T, T), bool), 1), -np.inf, s)
    m = s.max(-1, keepdims=True)
    e = np.exp(s - m)
    l = e.sum(-1, keepdims=True)
    return (e / l) @ v, (m + np.log(l))[..., 0]


def _inputs(B, H, T, d, seed):
    rng = np.random.default_rng(seed)
    return [rng.standard_normal((B, H, T, d)).astype(f32) for _ in range(3)]


def _run(gpu, q, k, v, causal):
    """O [B, H, T, d] and lse [B, H, T] of 128-query workgroups without a
    workspace, which never split the key range: the rule then takes the bf16
    matrix cores from T = 257 (full) and 385 (causal) on."""
    B, H, T, d = q.shape
    abi = Abi()
    try:
        pq, pk, pv = (abi.put(x) for x in (q, k, v))
        po, pl = abi.empty(B * H * T * d), abi.empty(B * H * T)
        st = (ctypes.c_int64 * 12)(*([H * T * d, T * d, d] * 4))
        abi.check(abi.L.aar_flash_fwd_strided_plan_f32(pq, pk, pv, po, pl, B, H, T, d, st, int(causal),
                                                       1.0 / math.sqrt(d), 128, None, 0, None))
        return abi.get(po, (B, H, T, d)).astype(np.float64), abi.get(pl, (B, H, T)).astype(np.float64)
    finally:
        abi.free()


def _close(got, ref):
    assert np.isfinite(got).all()
    top = np.abs(ref).max()  # keeps the norms' squares in range
    err = np.linalg.norm((got.reshape(ref.shape) - ref) / top) / np.linalg.norm(ref / top)
    assert err <= 5e-6, err


def _check(gpu, q, k, v, causal):
    for got, ref in zip(_run(gpu, q, k, v, causal), _exact(q, k, v, causal)):
        _close(got, ref)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("T", [257, 288, 385, 500])
@pytest.mark.parametrize("d", [36, 40, 64])
def test_head_dims_and_edges(gpu, d, T, causal):
    _check(gpu, *_inputs(1, 3, T, d, 1000 * d + T), causal)


def test_many_blocks(gpu):
    # more workgroups than the chip holds at once
    q, k, v = _inputs(60, 12, 400, 64, 3)
    o, lse = _run(gpu, q, k, v, True)
    for b in (0, 59):
        ro, rl = _exact(q[b:b + 1], k[b:b + 1], v[b:b + 1], True)
        _close(o[b:b + 1], ro)
        _close(lse[b:b + 1], rl)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [40, 56])
@pytest.mark.parametrize("scale_k,scale_v", [(1e-14, 1.0), (1e-20, 1.0), (1e-30, 1.0), (1e20, 1.0), (1e30, 1.0),
                                             (1.0, 1e-20), (1.0, 1e-30), (1.0, 1e25), (1.0, 1e36)])
def test_magnitudes(gpu, scale_k, scale_v, d, causal):
    q, k, v = _inputs(1, 3, 390, d, 5)
    _check(gpu, (q / f32(scale_k)).astype(f32), k * f32(scale_k), v * f32(scale_v), causal)


def test_one_tile_of_tiny_values(gpu):
    # the first tile's values lie far below the others': its queries see only them
    q, k, v = _inputs(1, 3, 400, 40, 6)
    v[:, :, :32] *= f32(1e-30)
    (o, _), (ro, _) = _run(gpu, q, k, v, True), _exact(q, k, v, True)
    _close(o[:, :, :32], ro[:, :, :32])
    _close(o[:, :, 32:], ro[:, :, 32:])


def test_tiny_row_seen_alone(gpu):
    # causal query 0 sees row 0 of V only, whose elements lie far below its
    # neighbours' in the same group of rows: O[0] is that row
    q, k, v = _inputs(1, 3, 400, 40, 8)
    rng = np.random.default_rng(8)
    v[:, :, 0] *= (10.0 ** -rng.uniform(30, 44, v[:, :, 0].shape)).astype(f32)
    o, _ = _run(gpu, q, k, v, True)
    # (P = 1 and l = 1 exactly; a normalisation may round once)
    np.testing.assert_allclose(o[:, :, 0], v[:, :, 0].astype(np.float64), rtol=2.0 ** -22, atol=2.0 ** -149)
    _close(o[:, :, 1:], _exact(q, k, v, True)[0][:, :, 1:])


def test_small_probabilities_read_out(gpu):
    # one row of V per column: O is the probabilities themselves, down to 2^-124.
    # |S| <= 130 ln 2 is summed over 36 products in fp32 (relative 2^-24 sqrt(36)
    # of it) and its exponential feels the absolute error: 130 ln 2 * 6 * 2^-24
    T, d = 300, 36
    q, k, v = _inputs(1, 2, T, d, 9)
    q *= f32(14.0)
    rows = 7 * np.arange(d)
    v[:] = 0.0
    v[:, :, rows, np.arange(d)] = 1.0
    o, _ = _run(gpu, q, k, v, False)
    ref = _exact(q, k, v, False)[0]
    small = (ref >= 2.0 ** -124) & (ref < 2.0 ** -105)
    assert small.sum() > 100
    keep = ref >= 2.0 ** -124
    assert (np.abs(o.reshape(ref.shape) - ref)[keep] <= 1e-4 * ref[keep]).all()


def test_tiny_scores(gpu):
    # causal query 0: lse is its one score, a product with a tiny element of K
    # that stands beside ordinary ones
    q, k, v = _inputs(1, 3, 400, 40, 10)
    q[:, :, 0] = 0.0
    q[:, :, 0, 5] = f32(2.0 ** 40)
    k[:, :, 0, 5] *= f32(2.0 ** -120)
    lse = _run(gpu, q, k, v, True)[1]
    want = 2.0 ** 40 * k[:, :, 0, 5].astype(np.float64) / math.sqrt(40)
    np.testing.assert_allclose(lse[:, :, 0], want, rtol=5e-7)


def _plain32(q, k, v, causal):
    """The formula in float32, for where it is not finite."""
    with np.errstate(all="ignore"):
        s = (q @ k.swapaxes(-1, -2)) * f32(1 / math.sqrt(q.shape[-1]))
        if causal:
            s = np.where(np.triu(np.ones(s.shape[-2:], bool), 1), f32(-np.inf), s)
        e = np.exp(s - s.max(-1, keepdims=True))
        return (e / e.sum(-1, keepdims=True)) @ v


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("where", ["q", "k", "v"])
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 3.4e38])
def test_not_finite(gpu, where, value, causal):
    """What a query sees of them, as plain float32 gives it.  Other heads, and the
    queries of earlier tiles under the causal mask, are untouched."""
    q, k, v = _inputs(1, 2, 400, 40, 7)
    clean = _exact(q, k, v, causal)[0]
    {"q": q, "k": k, "v": v}[where][0, 0, 40, 3] = value
    o, _ = _run(gpu, q, k, v, causal)
    _close(o[:, 1:], clean[:, 1:])
    got = o[0, 0]
    if where == "v":
        # column 3 alone, of the queries that see row 40 (the others of its tile
        # multiply it by zero)
        first = 40 if causal else 0
        hit = got[first:, 3]
        assert np.isnan(hit).all() if np.isnan(value) else ((hit > 1e30) if value > 0 else (hit < -1e30)).all()
        others = np.delete(got, 3, 1)
        _close(others[None], np.delete(clean[0, 0], 3, 1)[None])
        if causal:
            _close(got[:32], clean[0, 0, :32])
        return
    if causal:
        _close(got[:32 if where == "k" else 40], clean[0, 0, :32 if where == "k" else 40])
    want = _plain32(q, k, v, causal)[0, 0]
    bad = ~np.isfinite(want).all(-1)
    assert bad.any() and np.isnan(got[bad]).all()
    # (finite scores next to fp32's limit decide the softmax alone: 1e-5 of it)
    np.testing.assert_allclose(got[~bad], want[~bad], atol=1e-5, rtol=0)
