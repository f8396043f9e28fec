"""Row strides of the strided attention calls: the kernels address a staged
tile's rows by 32-bit byte offsets from its first one where those fit, which a
negative stride's (a sequence read backwards) do not.

On the CPU the offset arithmetic of csrc/hip/flash_offsets.hpp is compiled and
compared with 64-bit signed arithmetic; on the GPU operands laid out backwards
give, bit for bit, what the same operands laid out forwards give."""
from __future__ import annotations

import ctypes
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

from devutil import Abi

HIP_DIR = Path(__file__).resolve().parent.parent / "aar-vlm_amd" / "csrc" / "hip"

PROGRAM = r"""
#include "flash_offsets.hpp"
#include <cstdio>
int main() {
  using namespace aar;
  const int64_t k = int64_t(1) << 25;
  const int64_t strides[] = {-4 * k, -k, -k / 2, -4096, -64, -40, -4, -1, 0, 1, 4, 36, 64, 4096, k / 2, k - 1, k, 4 * k};
  for (int64_t st : strides) {
    const bool fit = tile_offsets_fit(st);
    if (fit != (st >= 0 && st < k)) return std::printf("stride %lld: fit %d\n", (long long)st, fit), 1;
    for (int row = 0; fit && row < 32; ++row)
      for (int col = 0; col < 128; ++col)
        if ((int64_t)tile_offset(row, st, col) != (row * st + col) * 4)
          return std::printf("stride %lld row %d col %d: %u\n", (long long)st, row, col, tile_offset(row, st, col)), 1;
  }
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_tile_offsets(tmp_path):
    src = tmp_path / "offsets.cpp"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", f"-I{HIP_DIR}", str(src), "-o", str(tmp_path / "offsets")], check=True)
    res = subprocess.run([str(tmp_path / "offsets")], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout


def test_staged_tiles_ask_for_the_rule():
    text = (HIP_DIR / "flash_attn.hip").read_text()
    assert text.count("small = tile_offsets_fit(st)") == text.count("small = ") == 2
    assert "Src s{base, st, {}, tile_offsets_fit(st)};" in text  # the DMA-staged tiles


def _forward(abi, q, k, v, causal, backwards):
    """O and lse; `backwards` lays every operand's rows out in reverse."""
    bh, T, d = q.shape
    flip = (lambda x: x[:, ::-1]) if backwards else (lambda x: x)
    last = 4 * (T - 1) * d if backwards else 0
    pq, pk, pv = (abi.put(flip(x)) + last for x in (q, k, v))
    po, pl = abi.empty(bh * T * d), abi.empty(bh * T)
    st = (ctypes.c_int64 * 12)(*([bh * T * d, T * d, -d if backwards else d] * 4))
    abi.check(abi.L.aar_flash_fwd_strided_plan_f32(pq, pk, pv, po + last, pl, 1, bh, T, d, st, int(causal),
                                                   1.0 / float(np.sqrt(d)), 128, None, 0, None))
    return flip(abi.get(po, (bh, T, d))), abi.get(pl, (bh, T))


@pytest.mark.gpu
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("T,d", [(257, 36), (390, 40), (500, 64), (512, 64)])
def test_forward_of_backward_rows(gpu, T, d, causal):
    # without a workspace nothing splits its key range
    rng = np.random.default_rng(T + d)
    q, k, v = (rng.standard_normal((6, T, d)).astype(np.float32) for _ in range(3))
    abi = Abi()
    try:
        for got, want in zip(_forward(abi, q, k, v, causal, True), _forward(abi, q, k, v, causal, False)):
            np.testing.assert_array_equal(got, want)
    finally:
        abi.free()


def _step(abi, ops, causal, query_block, key_block, fast, backwards):
    """O, lse, dQ, dK, dV on the paired 64-row plans (tiles staged by DMA) or
    the 128-row ones."""
    bh, T, d = ops[0].shape
    flip = (lambda x: x[:, ::-1]) if backwards else (lambda x: x)
    last = 4 * (T - 1) * d if backwards else 0
    L, s = abi.L, 1.0 / float(np.sqrt(d))
    pq, pk, pv, pdo = (abi.put(flip(x)) + last for x in ops)
    po, pl = abi.empty(bh * T * d) + last, abi.empty(bh * T)
    st = (ctypes.c_int64 * 24)(*([bh * T * d, T * d, -d if backwards else d] * 8))
    abi.check(L.aar_flash_fwd_strided_plan_f32(pq, pk, pv, po, pl, 1, bh, T, d, st, int(causal), s, query_block, None,
                                               0, None))
    wsb = (L.aar_flash_bwd_fast_workspace_bytes(bh, T, d, int(causal)) if fast
           else L.aar_flash_bwd_workspace_bytes(bh, T, d))
    grads = [abi.empty(bh * T * d) + last for _ in range(3)]
    abi.check(L.aar_flash_bwd_strided_plan_f32(pq, pk, pv, po, pl, pdo, *grads, 1, bh, T, d, st, int(causal), s,
                                               key_block, abi.alloc(wsb), wsb, None))
    return [flip(abi.get(p - last, (bh, T, d))) for p in (po, *grads)] + [abi.get(pl, (bh, T))]


@pytest.mark.gpu
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("fast", [False, True])
@pytest.mark.parametrize("block", [64, 128])
@pytest.mark.parametrize("T", [96, 300, 1056])
def test_step_of_backward_rows(gpu, T, block, fast, causal):
    rng = np.random.default_rng(T)
    ops = [rng.standard_normal((3, T, 64)).astype(np.float32) for _ in range(4)]
    abi = Abi()
    try:
        for got, want in zip(_step(abi, ops, causal, block, block, fast, True),
                             _step(abi, ops, causal, block, block, fast, False)):
            np.testing.assert_array_equal(got, want)
    finally:
        abi.free()
