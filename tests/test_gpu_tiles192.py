"""The tiled GEMMs on 192 x 256 work-groups (8 waves of 3 x 2 tiles, gemm_tiled.hip)
against the oracle bit for bit: 42 x 6 tiles, ragged both ways, one round of the CUs where
256 x 256 tiles leave a quarter idle."""
import numpy as np
import pytest

import synth
from gpu_util import from_dev, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("quant", ["q8_0", "q4_0"])
@pytest.mark.parametrize("nb,special", [
    (3, False),   # no full 4-block chunk: the tail alone
    (4, False),   # exactly one chunk: no DMA inside the fold
    (9, False),   # two chunks and a block
    (12, True),   # non-finite weight scales in the first, a middle and the last rows of waves
])
def test_gemm_tiles_192x256(hip, oracle, dev, quant, nb, special):
    nr, nc = 8000, 1500
    n, k = nb * 32, 18 if quant == "q4_0" else 34
    w = (synth.q4_0_matrix if quant == "q4_0" else synth.q8_0_matrix)(nr, n, 601, 0.02)
    a = synth.q8_0_matrix(nc, n, 602, 1.0)
    if special:
        for row, block, bits in ((0, 0, 0x7C00), (95, 5, 0xFC00), (96, 4, 0x7E00), (191, 11, 0x7C00),
                                 (192 + 64, 7, 0x7C00), (7999, 8, 0xFC00), (500, 3, 0x0001)):
            w.reshape(nr, nb, k)[row, block, :2] = np.frombuffer(np.uint16(bits).tobytes(), np.uint8)
    dw, da = to_dev(w, dev), to_dev(a, dev)
    tx = to_dev(np.zeros(hip.gemm_tiles_bytes(nr, nb), np.uint8), dev)
    ty = to_dev(np.zeros(hip.gemm_tiles_bytes(nc, nb), np.uint8), dev)
    (hip.pack_q4_0_to_gemm_tiles if quant == "q4_0" else hip.pack_q8_0_to_gemm_tiles)(
        nr, nb, dw, w.shape[1], tx)
    hip.pack_q8_0_to_gemm_tiles(nc, nb, da, a.shape[1], ty)
    bs = nc + 3
    s = to_dev(np.full(nr * bs, -7.0, np.float32), dev)
    (hip.q4_0_q8_0_gemm_tiles if quant == "q4_0" else hip.q8_0_q8_0_gemm_tiles)(
        n, s, tx, ty, nr, nc, bs)
    want = (oracle.gemm_q4_0 if quant == "q4_0" else oracle.gemm_q8_0)(
        n, w, a, a.shape[1], nr, nc, w.shape[1], bs, 16).reshape(nr, bs)[:, :nc]
    got = from_dev(s).reshape(nr, bs)
    assert np.all(got[:, nc:] == -7.0)
    got = got[:, :nc]
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(got[~nan].view(np.uint32), want[~nan].view(np.uint32))
