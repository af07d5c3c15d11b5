"""Which kernel an entry runs at a size: the shipped rules, replayed without a GPU
(tests/launches.py)."""
import random

import pytest

import launches
import tcrv_hip

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
    ("q4_0", 15568, 33, 6656, "pack_tiles_ranges2<true, 2, true>"),
    ("q8_0", 4096, 4096, 4096, "pack_tiles_ranges2<false, 2, false>"),  # 1024 ranges of weights
    ("q8_0", 4032, 4096, 4096, "pack_tiles_ranges2<false, 1, false>"),  # 1008
    ("q8_0", 3001, 4096, 2912, "pack_tiles_ranges2<false, 1, false>"),
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


def workspace_needed(quant, nr, nc, n, xpad, ypad):
    """What include/tcrv_hip.h says of the workspace entries."""
    nb = n // 32
    bx, by = nb * (18 if quant == "q4_0" else 34) + xpad, nb * 34 + ypad

    def aligned(k):
        return bx % k == 0 and by % k == 0

    def tiles(k):
        return -(-nr // k) * -(-nc // k)

    if nr < 256 or nc < 2 or nb < 1:
        return False
    if nc <= 24 and nb % 2 == 0 and aligned(4):
        return False
    return not (nb % 8 == 0 and nb <= 128 and aligned(16) and tiles(32) > 256 and tiles(64) <= 448)


@pytest.mark.parametrize("quant", ["q4_0", "q8_0"])
def test_workspace_is_required_where_the_header_says(quant):
    """A missing workspace is refused exactly there, and nothing is launched; elsewhere the call
    runs.  What a call writes into it is unspecified (few outputs: nothing)."""
    rng = random.Random(5)
    sizes = [(255, 64, 4096, 0, 0), (256, 1, 4096, 0, 0), (256, 2, 32, 0, 0), (256, 24, 4096, 0, 0),
             (256, 25, 4096, 0, 0), (256, 24, 4096 + 32, 0, 0), (256, 24, 4096, 2, 0),
             (4096, 128, 4096, 0, 0), (4096, 128, 4352, 0, 0), (4096, 128, 4096, 4, 0),
             (4096, 448, 4096, 0, 0), (4096, 449, 4096, 0, 0), (512, 512, 4096, 0, 0),
             (512, 544, 4096, 0, 0)]
    sizes += [(rng.randint(200, 6000), rng.randint(1, 600), 32 * rng.randint(1, 140),
               rng.choice((0, 0, 2, 4, 16)), rng.choice((0, 0, 2, 16))) for _ in range(200)]
    calls = []
    for nr, nc, n, xpad, ypad in sizes:
        name, args = launches.gemm_call(quant, "ws", nr, nc, n, xpad, ypad)
        calls.append((name, args[:-2] + (0, 0)))
    for size, (status, xs) in zip(sizes, launches.replay(calls)):
        want = tcrv_hip.ERR_NULL_POINTER if workspace_needed(quant, *size) else 0
        assert status == want and bool(xs) == (want == 0), (size, status, xs)
