"""The forward on the bf16 matrix cores (operands in three bf16 parts) against
float64: head dims that fill and half fill the padded width,
sequences at the edges of tiles and blocks past the lengths that keep the fp32
instruction, and magnitudes that the split hands
to the fp32 instruction.  Bound on the relative 2-norm error of O and lse:
5e-6, the rounding of fp32 sums over d <= 64 products in S (at most about
sqrt(64) 2^-24 |S| ~ 2e-6 of P at |S| <= 4) and of O's over the keys (3e-7)."""
from __future__ import annotations

import math

import numpy as np
import pytest

from devutil import dev, host

pytestmark = pytest.mark.gpu
f32 = np.float32
# causal grids of at most 256 workgroups would split the key range instead
HEADS = {False: (1, 3), True: (7, 10)}


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
    o, lse = gpu._core._flash_attention_fwd(dev(gpu, q), dev(gpu, k), dev(gpu, v), causal)
    return host(gpu, o).astype(np.float64), host(gpu, lse).astype(np.float64)


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
    _check(gpu, *_inputs(*HEADS[causal], T, d, 1000 * d + T), causal)


def test_many_blocks(gpu):
    # causal d = 64 above the grids that take 64-query workgroups
    q, k, v = _inputs(60, 12, 400, 64, 3)
    o, lse = _run(gpu, q, k, v, True)
    for b in (0, 59):
        ro, rl = _exact(q[b:b + 1], k[b:b + 1], v[b:b + 1], True)
        _close(o[b:b + 1], ro)
        _close(lse.reshape(60, 12, 400)[b:b + 1], rl)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [40, 56])
@pytest.mark.parametrize("scale_k,scale_v", [(1e-14, 1.0), (1e-20, 1.0), (1e-30, 1.0), (1e20, 1.0), (1e30, 1.0),
                                             (1.0, 1e-20), (1.0, 1e-30), (1.0, 1e25), (1.0, 1e36)])
def test_magnitudes(gpu, scale_k, scale_v, d, causal):
    q, k, v = _inputs(*HEADS[causal], 390, d, 5)
    _check(gpu, (q / f32(scale_k)).astype(f32), k * f32(scale_k), v * f32(scale_v), causal)


def test_one_tile_of_tiny_values(gpu):
    # the first tile's values lie far below the others': its queries see only them
    q, k, v = _inputs(7, 10, 400, 40, 6)
    v[:, :, :32] *= f32(1e-30)
    (o, _), (ro, _) = _run(gpu, q, k, v, True), _exact(q, k, v, True)
    _close(o[:, :, :32], ro[:, :, :32])
    _close(o[:, :, 32:], ro[:, :, 32:])


@pytest.mark.parametrize("where", ["q", "k", "v"])
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 3.4e38])
def test_not_finite(gpu, where, value):
    # what a query sees of them, as plain float32 gives it; other heads are untouched
    q, k, v = _inputs(1, 2, 300, 40, 7)
    {"q": q, "k": k, "v": v}[where][0, 0, 40, 3] = value
    o, _ = _run(gpu, q, k, v, False)
    _close(o[:, 1:], _exact(q[:, 1:], k[:, 1:], v[:, 1:], False)[0])
    if where == "v":
        hit = o[0, 0, :, 3]
        assert np.isnan(hit).all() if np.isnan(value) else ((hit > 1e30) if value > 0 else (hit < -1e30)).all()
    elif where == "q" and value != f32(3.4e38):
        assert np.isnan(o[0, 0, 40]).all() and np.isfinite(np.delete(o[0, 0], 40, 0)).all()
