"""CPU checks of the f32 tiles: the LDS layout of a 64-column bf16 plane
(f32_btr64_offset), the rule that picks the 64 x 64 tiles (tile_shape), and
the bound of the partial products that the bf16 split leaves out."""
from __future__ import annotations

import subprocess
from pathlib import Path

import numpy as np
import pytest

from welder_typical_chain_amd import _lib

ROOT = Path(__file__).resolve().parents[1]

SOURCE = r"""
#include <cstdio>
#include <set>
#include "tile_layout.h"
using namespace wtc;
int main() {
  std::set<int> bytes;  // every value of the plane at a place of its own
  for (int k = 0; k < 32; ++k)
    for (int n = 0; n < 64; ++n) {
      const int o = f32_btr64_offset(k, n);
      if (o < 0 || o + 2 > 64 * 64 || !bytes.insert(o).second) return std::puts("place"), 1;
      if ((n & 7) && f32_btr64_offset(k, n - 1) + 2 != o) return std::puts("chunk"), 1;
    }
  for (int s = 0; s < 2; ++s)
    for (int h = 0; h < 2; ++h)
      for (int nb = 0; nb < 64; nb += 32)
        for (int half = 0; half < 64; half += 32) {  // 32 lanes of a transpose read: 256 bytes
          std::set<int> banks;
          for (int l = half; l < half + 32; ++l)
            for (int b = 0; b < 8; b += 4)
              if (!banks.insert((f32_btr64_offset(btr_k(s, h, l), btr_n(nb, l)) + b) / 4 % 64).second)
                return std::puts("bank"), 1;
        }
  return std::puts("OK"), 0;
}
"""


def test_plane_of_64_columns(tmp_path):
    src = tmp_path / "f32_layout.cpp"
    src.write_text(SOURCE)
    exe = tmp_path / "f32_layout"
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", f"-I{ROOT / 'welder_typical_chain_amd' / 'csrc'}",
                    str(src), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0 and res.stdout.strip() == "OK", res.stdout


@pytest.mark.parametrize("batch,m,n,k,path,grid", [
    (1, 128, 128, 128, _lib.PATH_EXCHANGE, 4),       # 64 x 64
    (1, 1024, 1024, 1024, _lib.PATH_EXCHANGE, 256),
    (1, 2048, 1024, 512, _lib.PATH_EXCHANGE, 512),   # two to a CU
    (1, 2049, 1024, 512, _lib.PATH_EXCHANGE, 136),   # 528 of 64: 128 x 128
    (1, 64, 4096, 512, _lib.PATH_EXCHANGE, 64),
    (1, 64, 4104, 512, _lib.PATH_EXCHANGE, 33),      # 65 column tiles of 64
    (1, 1024, 1024, 1024, _lib.PATH_SPLIT, 64),      # split and unfused: 128 x 128
    (1, 1024, 1024, 1024, _lib.PATH_UNFUSED, 64),
])
def test_tile_rule(native_lib, batch, m, n, k, path, grid):
    pl = _lib.plan(batch, m, n, k, _lib.DTYPE_F32, _lib.DTYPE_F32, path)
    assert pl["grid"] == grid and pl["path"] == path
    # every tile of the exchange path has its slot in the workspace
    if path == _lib.PATH_EXCHANGE:
        assert pl["workspace_bytes"] >= 256 + 4096 + grid * 1024


def _bf16(x):
    """x (f32) rounded to bf16, to nearest even, as f32."""
    u = x.view(np.uint32)
    return ((u + 0x7FFF + ((u >> 16) & 1)) & 0xFFFF0000).astype(np.uint32).view(np.float32)


def test_bound_of_the_products_left_out():
    """Over every mantissa: x0 + x1 + x2 is x, and a1 b2 + a2 b1 + a2 b2 of any two
    values is at most 2^-24 + 2^-34 of their product, nearly reached; over random
    pairs its mean square is below 2^-27 and its sign even."""
    x = (np.arange(2 ** 23, dtype=np.uint32) | 0x3F800000).view(np.float32)
    x0 = _bf16(x)
    x1 = _bf16(x - x0)
    x2 = x - x0 - x1
    assert np.array_equal(_bf16(x2), x2)
    assert np.array_equal(x0.astype(np.float64) + x1 + x2, x.astype(np.float64))
    r1, r2 = x1.astype(np.float64) / x, x2.astype(np.float64) / x
    most1, most2 = np.abs(r1).max(), np.abs(r2).max()
    assert 2 * most1 * most2 + most2 ** 2 <= 2.0 ** -24 + 2.0 ** -34
    worst = np.abs(2 * r1 * r2 + r2 * r2)
    assert worst.max() > 2.0 ** -24.02 and abs(float(x[worst.argmax()]) - 1.0039) < 1e-4
    rng = np.random.default_rng(1)
    i, j = (rng.integers(0, x.size, 1_000_000) for _ in range(2))
    out = r1[i] * r2[j] + r2[i] * r1[j] + r2[i] * r2[j]
    assert np.sqrt(np.mean(out ** 2)) < 2.0 ** -27 and abs(out.mean()) < 2.0 ** -35
