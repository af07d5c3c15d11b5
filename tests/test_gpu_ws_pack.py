"""The workspace entries' pack with the weights' ranges in pairs (gemm_tiled.hip), through the
entries against the oracle bit for bit."""
import numpy as np
import pytest

import launches
import synth
from gpu_util import assert_f32_parity, from_dev, to_dev

SIZES = [
    # nr, nc, nb, weight pad, token pad
    (65537, 25, 8, 0, 0),  # 1025 ranges: the last work-group has one
    (32769, 27, 9, 0, 2),  # 1026, every second one block long; 2-byte aligned rows
    (32800, 33, 15, 2, 0),
]


@pytest.mark.parametrize("nr,nc,nb,xpad,ypad", SIZES)
@pytest.mark.parametrize("quant", ["q4_0", "q8_0"])
def test_packs_in_pairs(quant, nr, nc, nb, xpad, ypad):
    names = launches.kernels([launches.gemm_call(quant, "ws", nr, nc, nb * 32, xpad, ypad)])[0]
    assert names[0] == f"pack_tiles_ranges2<{'true' if quant == 'q4_0' else 'false'}, 2>"


@pytest.mark.gpu
@pytest.mark.parametrize("nr,nc,nb,xpad,ypad", SIZES)
@pytest.mark.parametrize("quant", ["q4_0", "q8_0"])
def test_parity(hip, oracle, dev, quant, nr, nc, nb, xpad, ypad):
    q4, n = quant == "q4_0", nb * 32
    w = np.pad((synth.q4_0_matrix if q4 else synth.q8_0_matrix)(nr, n, 821, 0.02),
               ((0, 0), (0, xpad)))
    a = np.pad(synth.q8_0_matrix(nc, n, 822, 1.0), ((0, 0), (0, ypad)))
    size = hip.q8_0_q8_0_gemm_workspace_bytes(n, nr, nc)
    s = to_dev(np.full(nr * nc, -7.0, np.float32), dev)
    (hip.q4_0_q8_0_gemm_ws if q4 else hip.q8_0_q8_0_gemm_ws)(
        n, s, to_dev(w, dev), to_dev(a, dev), a.shape[1], nr, nc, w.shape[1], nc,
        to_dev(np.full(size, 0xEE, np.uint8), dev), size)
    want = (oracle.gemm_q4_0 if q4 else oracle.gemm_q8_0)(
        n, w, a, a.shape[1], nr, nc, w.shape[1], nc, 8)
    assert_f32_parity(from_dev(s), want, what=f"{quant} {nr}x{nc}x{n}")
