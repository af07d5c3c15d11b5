"""The work-group order of the plain-row and repack GEMMs over the 8 XCDs (csrc/tile_order.h):
every tile once, the XCDs' runs within one tile of each other or one work-group a CU at most,
the launched grids as long as the longest run, and (-m gpu) grids of several z against the oracle."""
import os
import subprocess

import numpy as np
import pytest

import launches
import synth
from gpu_util import assert_f32_parity, from_dev, to_dev

CSRC = os.path.join(launches.ROOT, "tianchen-rv_amd", "csrc")

CHECK = r"""
#include "tile_order.h"
#include <cstdio>
#include <vector>
int main() {
  using namespace tcrv;
  unsigned r, t;
  while (std::scanf("%u %u", &r, &t) == 2) {
    TileOrder o;
    if (!tile_order(r, t, &o)) return 1;
    std::vector<char> seen(static_cast<size_t>(r) * t);
    size_t most = 0, least = ~static_cast<size_t>(0);
    for (unsigned x = 0; x < kXcds; ++x) {
      size_t live = 0;
      for (unsigned z = 0; z < o.slots_z; ++z)
        for (unsigned y = 0; y < o.slots_y; ++y) {
          const TilePos p = xcd_tile(o.units, r, t, o.inv, x, y, z);
          if (!p.live) continue;
          ++live;
          if (p.tm >= r || p.tn >= t || seen[static_cast<size_t>(p.tm) * t + p.tn]++) return 2;
        }
      most = live > most ? live : most;
      least = live < least ? live : least;
    }
    for (char c : seen)
      if (!c) return 3;
    // even runs, or whole row tiles on at most one work-group a CU
    if (most - least > 1 && (most > kXcdCus || most % t)) return 4;
  }
  TileOrder o;
  if (!tile_order(1, kMaxTiles - 1, &o) || o.slots_z > 65535) return 5;
  return tile_order(kMaxTiles / 2, 2, &o) || tile_order(1, kMaxTiles, &o) ? 6 : 0;
}
"""


def test_every_tile_once_and_balanced(tmp_path):
    src, exe = tmp_path / "check.cpp", tmp_path / "check"
    src.write_text(CHECK)
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", f"-I{CSRC}", str(src), "-o",
                    str(exe)], check=True)
    pairs = [(r, t) for r in (1, 2, 3, 7, 8, 9, 16, 35, 64, 71) for t in range(1, 66)]
    pairs += [(1, 100003), (100003, 1), (3, 65537), (4099, 33), (257, 1021), (2, 1 << 20)]
    out = subprocess.run([str(exe)], input="\n".join(f"{r} {t}" for r, t in pairs), text=True)
    assert out.returncode == 0


# the row and token extent of a work-group's tile
TILES = {"gemm_batch": lambda a: (16, 16), "gemm_batch_one": lambda a: (16, 16),
         "gemm_rows16": lambda a: (16 * int(a[1]), 32),
         "gemm_repack_mid": lambda a: (32 * int(a[0]), 32 * int(a[1]))}


@pytest.mark.parametrize("quant,entry,nr,nc,n,kernel", [
    ("q8_0", "plain", 2220, 219, 2304, "gemm_rows16"),  # 35 x 7 tiles
    ("q8_0", "plain", 64, 8192, 4096, "gemm_rows16"),   # one row tile
    ("q4_0", "plain", 576, 896, 4096, "gemm_rows16"),   # nine
    ("q8_0", "ws", 1170, 327, 12608, "gemm_rows16"),
    ("q4_0", "plain", 16, 4096, 4096, "gemm_batch"),    # one row tile, 256 token groups
    ("q8_0", "plain", 2, 319, 12064, "gemm_batch"),
    ("q4_0", "plain", 4096, 16, 4096, "gemm_batch_one"),
    ("q8_0", "plain", 4100, 2, 2912, "gemm_batch_one"),
    ("q4_0", "repack", 2176, 768, 4096, "gemm_repack_mid"),  # 17 x 12
    ("q4_0", "repack", 512, 4096, 4096, "gemm_repack_mid"),
    ("q4_0", "repack", 1152, 1088, 4096, "gemm_repack_mid"),
])
def test_no_xcd_gets_more_than_its_share(quant, entry, nr, nc, n, kernel):
    (status, xs), = launches.replay([launches.gemm_call(quant, entry, nr, nc, n)])
    assert status == 0 and len(xs) == 1
    name, args = xs[0].name.rstrip(">").split("<")
    assert name == kernel
    rows, toks = TILES[name](args.split(", "))
    total = -(-nr // rows) * -(-nc // toks)
    gx, gy, gz = xs[0].grid
    assert gx == 8 and gy * gz <= max(-(-total // 8), 32)


@pytest.mark.gpu
@pytest.mark.parametrize("quant", ["q4_0", "q8_0"])
@pytest.mark.parametrize("nr,nc,nb,xpad", [
    (16, 65700, 1, 0),   # gemm_batch: 4107 token groups of one row tile, 514 slots an XCD
    (8200, 1020, 1, 2),  # gemm_rows16: 129 x 32 tiles, 516 slots
])
def test_grids_of_several_z(hip, oracle, dev, quant, nr, nc, nb, xpad):
    n = nb * 32
    w = np.pad((synth.q4_0_matrix if quant == "q4_0" else synth.q8_0_matrix)(nr, n, 801, 0.02),
               ((0, 0), (0, xpad)))
    a = synth.q8_0_matrix(nc, n, 802, 1.0)
    s = to_dev(np.full(nr * nc, -7.0, np.float32), dev)
    run = hip.q4_0_q8_0_gemm if quant == "q4_0" else hip.q8_0_q8_0_gemm
    run(n, s, to_dev(w, dev), to_dev(a, dev), a.shape[1], nr, nc, w.shape[1], nc)
    want = (oracle.gemm_q4_0 if quant == "q4_0" else oracle.gemm_q8_0)(
        n, w, a, a.shape[1], nr, nc, w.shape[1], nc, 8)
    assert_f32_parity(from_dev(s), want, what=f"{quant} {nr}x{nc}x{n}")
