"""Every GEMM kernel at a ragged size that reaches it, with a part chunk at the end of K, under
ordinary and special scales.  That a size reaches its kernel is replayed through the library's own
rules without a GPU; the outputs (-m gpu) are compared with the oracle bit for bit, on sampled rows
where the size is large."""
import re
import subprocess

import numpy as np
import pytest
import torch

import launches
import synth
from gpu_util import assert_f32_parity, assert_f32_parity_nan, empty_dev, from_dev, to_dev
from test_gpu_special import _set_scale, _x16_source, q4, q8

Q = {"q4_0": "true", "q8_0": "false"}


def both(kernel, *size):
    return [(kernel.replace("%", Q[quant]), quant) + size for quant in ("q4_0", "q8_0")]


# kernel, quant, entry, weight rows, tokens, blocks, weight pad, token pad
SIZES = [s for quant in ("q4_0", "q8_0") for s in [
    (f"gemv_{quant}_q8_0_cols<2, true>", quant, "plain", 37, 2, 128, 0, 0),
    (f"gemv_{quant}_q8_0_cols<2, false>", quant, "plain", 37, 2, 258, 4, 8),
    (f"gemv_{quant}_q8_0_cols<4, true>", quant, "plain", 37, 3, 128, 0, 0),
    (f"gemv_{quant}_q8_0_cols<4, false>", quant, "plain", 37, 4, 258, 0, 4),
]]
SIZES += both("gemm_batch<%, 8, false>", "plain", 300, 30, 67 + 64, 0, 0)
SIZES += both("gemm_batch<%, 16, false>", "plain", 300, 30, 67, 2, 0)
SIZES += both("gemm_batch_one<%, 8>", "plain", 300, 15, 67 + 64, 0, 0)
SIZES += both("gemm_batch_one<%, 16>", "plain", 300, 15, 67, 2, 0)
SIZES += both("gemm_rows16<%, 2>", "plain", 2100, 66, 33, 0, 2)
SIZES += both("gemm_rows16<%, 4>", "plain", 2100, 130, 22, 2, 0)
SIZES += both("gemm_rows_few<%>", "plain", 1000, 800, 24, 0, 16)
for nb, ypad in ((2, 0), (8, 4), (10, 4)):  # 4-block chunks: none, two whole, a part one
    SIZES += both("gemm_wide<%>", "plain", 2100, 1000, nb, 0, ypad)
SIZES += both("gemm_wide<%>", "plain", 2100, 1000, 42, 4, 0)
for nb, xpad in ((2, 0), (8, 4), (10, 0)):
    SIZES += [("gemm_occ<true>", "q4_0", "plain", 200, 6190, nb, xpad, 0),
              ("gemm_occ<false>", "q8_0", "plain", 200, 5930, nb, xpad, 0)]
SIZES += both("gemm_tiles16<%>", "tiles", 300, 200, 9, 0, 0)
SIZES += both("gemm_tiles32<%>", "tiles", 1000, 700, 9, 0, 0)
for q in ("q4_0", "q8_0"):
    for nb in (5, 6, 13):  # 6-block chunks: none, one whole, a part one
        SIZES.append(("gemm_tiles_q4" if q == "q4_0" else "gemm_tiles_q8<true>", q, "tiles", 3100,
                      2100, nb, 0, 0))
    SIZES += [(f"gemm_tiles256_{q[:2]}<Wave2x4>", q, "tiles", 3400, 3700, 13, 0, 0),
              (f"gemm_tiles256_{q[:2]}<Wave3x2>", q, "tiles", 4000, 2900, 13, 0, 0)]
# x16 weights: weight rows a multiple of 16, tokens of 4; the pad is of the output rows
SIZES += [("gemm_repack_q4_0", "q4_0", "repack", 2064, 2052, 9, 0, 0),
          ("gemm_repack_q4_0", "q4_0", "repack", 2064, 2052, 21, 3, 0)]  # scalar stores
IDS = [f"{s[0]}-{s[5]}" for s in SIZES]


def test_sizes_reach_their_kernels():
    calls = [launches.gemm_call(quant, entry, nr, nc, nb * 32, xpad, ypad)
             for _, quant, entry, nr, nc, nb, xpad, ypad in SIZES]
    for size, names in zip(SIZES, launches.kernels(calls)):
        assert names == [size[0]], size


def test_every_gemm_kernel_is_reached():
    """No GEMM kernel of the library is without a size here (the packs, the codecs and the decode
    GEMVs have theirs elsewhere; the batch kernel's 64-bit form and repack_mid too)."""
    out = subprocess.run(["nm", "-DC", "--defined-only", launches.LIB], capture_output=True,
                         text=True, check=True).stdout
    have = set(re.findall(r"tcrv::(gem[mv]_\w+(?:<[^>]*>)?)\(", out.replace("tcrv::Wave", "Wave")))
    have = {k for k in have if k.startswith("gemm_") or "_cols" in k}
    elsewhere = {k for k in have if k.startswith(("gemm_repack_mid<", "gemm_batch<"))
                 and k not in {s[0] for s in SIZES}}
    assert have - elsewhere == {s[0] for s in SIZES}


def operands(quant, entry, nr, nc, nb, special):
    w = (q4(nr, nb, 841, nonfinite_every=16 if special == "spread" else 0) if quant == "q4_0" else
         q8(nr, nb, 841, 0.02, nonfinite_every=16 if special == "spread" else 0))
    a = q8(nc, nb, 842, 1.0, nonfinite_every=37 if special else 0)
    planted = [min(nr - 1, max(1, nr * k // 7)) for k in range(1, 7)]
    if special == "planted":  # one bad scale a row: in the first, a middle and the last blocks
        blk = 18 if quant == "q4_0" else 34
        at = (nb // 2, 0, nb - 1, nb - 2, nb // 2, nb * 2 // 3)
        for r, b, bits in zip(planted, at, (0x7C00, 0xFC00, 0x7E00, 0x7C00, 0xFC00, 0x0001)):
            _set_scale(w, r, b, blk, bits)
        r, b = planted[4], at[4]  # an infinite scale over a zero block sum: NaN
        w[r, b * blk + 2:(b + 1) * blk] = 0x88 if quant == "q4_0" else 0
    return w, a, planted


@pytest.mark.gpu
@pytest.mark.parametrize("special", ["", "spread", "planted"])
@pytest.mark.parametrize("kernel,quant,entry,nr,nc,nb,xpad,ypad", SIZES, ids=IDS)
def test_parity(hip, oracle, dev, kernel, quant, entry, nr, nc, nb, xpad, ypad, special):
    print(f"{kernel} {nr} x {nc} x {nb} blocks, {special or 'ordinary'} scales", flush=True)
    n = nb * 32
    if special:
        w, a, planted = operands(quant, entry, nr, nc, nb, special)
    else:
        w = (synth.q4_0_matrix if quant == "q4_0" else synth.q8_0_matrix)(nr, n, 841, 0.02)
        a, planted = synth.q8_0_matrix(nc, n, 842, 1.0), []
    if entry == "repack":
        bs = nr + xpad
        packed = oracle.pack_q4_0x16(_x16_source(w, nb, 18), nr // 16 * nb)
        ax4 = oracle.pack_q8_0x4(a, nc, nb, a.shape[1])
        s = to_dev(np.full(nc * bs, -7.0, np.float32), dev)
        hip.repack_gemm_q4_0_q8_0(n, s, to_dev(packed, dev), to_dev(ax4, dev), nc, nr, bs)
        got = from_dev(s).reshape(nc, bs)
        assert np.all(got[:, nr:] == -7.0)
        want = oracle.repack_gemm_q4_0(n, packed, ax4, nc, nr, bs).reshape(nc, bs)[:, :nr]
        assert_f32_parity_nan(got[:, :nr], want, what=kernel)
        return
    w, a = np.pad(w, ((0, 0), (0, xpad))), np.pad(a, ((0, 0), (0, ypad)))
    bs = nc + 3
    s = to_dev(np.full(nr * bs, -7.0, np.float32), dev)
    if entry == "plain":
        getattr(hip, f"{quant}_q8_0_gemm")(n, s, to_dev(w, dev), to_dev(a, dev), a.shape[1], nr, nc,
                                           w.shape[1], bs)
    else:
        tx = empty_dev(hip.gemm_tiles_bytes(nr, nb), torch.uint8, dev)
        ty = empty_dev(hip.gemm_tiles_bytes(nc, nb), torch.uint8, dev)
        getattr(hip, f"pack_{quant}_to_gemm_tiles")(nr, nb, to_dev(w, dev), w.shape[1], tx)
        hip.pack_q8_0_to_gemm_tiles(nc, nb, to_dev(a, dev), a.shape[1], ty)
        getattr(hip, f"{quant}_q8_0_gemm_tiles")(n, s, tx, ty, nr, nc, bs)
    got = from_dev(s).reshape(nr, bs)
    assert np.all(got[:, nc:] == -7.0)
    # a row of every residue of the kernels' row tiles, and what was planted
    rows = np.unique(np.clip([0, 1, nr - 1, nr - 2] + [r + d for r in planted for d in (-1, 0, 1)] +
                             list(range(5, nr, 67)), 0, nr - 1))
    want = (oracle.gemm_q4_0 if quant == "q4_0" else oracle.gemm_q8_0)(
        n, np.ascontiguousarray(w[rows]), a, a.shape[1], len(rows), nc, w.shape[1], nc, 8)
    check = assert_f32_parity_nan if special else assert_f32_parity
    check(got[rows][:, :nc], want, what=f"{kernel} {nr}x{nc}x{n}")
    if special == "planted":
        want = want.reshape(len(rows), nc)
        assert np.isinf(want[rows == planted[0]]).any() and np.isnan(want[rows == planted[4]]).all()
