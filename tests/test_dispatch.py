"""Which kernel an entry runs at a size: the shipped rules, replayed without a GPU
(tests/launches.py)."""
import pytest

import launches

# quant, entry, weight rows, tokens, n, keyword arguments of gemm_call, kernel
SIZES = [
    # half-empty 64-row tiles: as many 32-row work-groups
    ("q8_0", "plain", 31, 9893, 3840, {}, "gemm_rows16<false, 2>"),
    ("q4_0", "plain", 2317, 211, 4960, {}, "gemm_rows16<true, 2>"),
    ("q8_0", "plain", 212, 4169, 2176, {}, "gemm_rows16<false, 2>"),
    ("q4_0", "plain", 4096, 128, 4096, {}, "gemm_rows16<true, 4>"),
    ("q8_0", "plain", 4096, 64, 4096, {}, "gemm_rows16<false, 2>"),
    # few outputs, where gemm_rows_few serves
    ("q4_0", "plain", 4096, 192, 4096, {}, "gemm_rows16<true, 2>"),
    ("q8_0", "plain", 4096, 192, 4096, {}, "gemm_rows16<false, 2>"),
    ("q8_0", "plain", 4096, 192, 4352, {}, "gemm_rows_few<false>"),
    ("q8_0", "plain", 6457, 75, 512, {}, "gemm_rows16<false, 2>"),
    ("q8_0", "plain", 4894, 127, 256, {}, "gemm_rows_few<false>"),
    ("q4_0", "plain", 1166, 596, 256, {}, "gemm_rows_few<true>"),
    ("q8_0", "plain", 18006, 21, 1792, {}, "gemm_rows16<false, 2>"),
    ("q4_0", "plain", 790, 1238, 3584, {}, "gemm_rows16<true, 4>"),
    # few weight rows and many tokens, K no multiple of 256
    ("q8_0", "plain", 190, 8881, 10432, {}, "gemm_occ<false>"),
    ("q4_0", "plain", 120, 14581, 960, {}, "gemm_occ<true>"),
    ("q8_0", "plain", 154, 7280, 2880, {}, "gemm_rows16<false, 2>"),
    # against the 256-row tiles
    ("q8_0", "plain", 6192, 244, 640, {}, "gemm_wide<false>"),
    ("q4_0", "plain", 977, 1672, 320, {}, "gemm_rows16<true, 4>"),
    ("q8_0", "plain", 732, 1379, 640, {}, "gemm_rows16<false, 2>"),
    ("q4_0", "plain", 4096, 512, 4160, {}, "gemm_rows16<true, 4>"),
    ("q4_0", "plain", 4096, 1000, 4160, {}, "gemm_wide<true>"),
]


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "-".join(map(str, s[:5])))
def test_kernel_of_a_size(size):
    *call, kw, want = size
    assert launches.kernels([launches.gemm_call(*call, **kw)])[0][-1] == want


@pytest.mark.parametrize("quant,nr,nc,n,want", [
    ("q4_0", 15568, 33, 6656, "pack_tiles_ranges2<true, 2>"),
    ("q8_0", 4096, 4096, 4096, "pack_tiles_ranges2<false, 2>"),  # 1024 ranges of weights
    ("q8_0", 4032, 4096, 4096, "pack_tiles_ranges2<false, 1>"),  # 1008
    ("q8_0", 3001, 4096, 2912, "pack_tiles_ranges2<false, 1>"),
])
def test_pack_of_a_workspace_gemm(quant, nr, nc, n, want):
    assert launches.kernels([launches.gemm_call(quant, "ws", nr, nc, n)])[0][0] == want


@pytest.mark.parametrize("quant,rows,nb,bx,want", [
    ("q8_0", 4037, 11, 11 * 34, "pack_gemm_tiles"),                       # 128 ranges
    ("q4_0", 1513, 12, 12 * 18, "pack_q4_tiles"),
    ("q8_0", 4161, 16, 16 * 34 + 2, "pack_tiles_ranges<false, 1, false>"),  # 132, unaligned
    ("q4_0", 4161, 9, 9 * 18, "pack_tiles_ranges<true, 1, false>"),
    ("q8_0", 333, 16, 16 * 34, "pack_tiles_ranges<false, 1, true>"),      # few, but whole and aligned
    ("q8_0", 24577, 9, 9 * 34, "pack_tiles_ranges<false, 2, false>"),
    ("q4_0", 11008, 128, 128 * 18, "pack_q4_tiles_span"),
])
def test_kernel_of_a_pack(quant, rows, nb, bx, want):
    call = f"tcrv_hip_pack_{quant}_to_gemm_tiles", (rows, nb, launches.X, bx, launches.WS)
    assert launches.kernels([call]) == [[want]]
