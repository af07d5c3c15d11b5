"""The workspace entries' pack (gemm_tiled.hip): the weights' ranges in pairs, and their row groups
going round the XCDs, through the entries against the oracle bit for bit."""
import numpy as np
import pytest

import launches
import synth
from gpu_util import assert_f32_parity, from_dev, to_dev

SIZES = [
    # nr, nc, nb, weight pad, token pad, ranges a work-group, work-groups of a row group or 0: in order
    (65537, 25, 8, 0, 0, 2, 0),   # 1025 ranges: the last work-group has one
    (32769, 27, 9, 0, 2, 2, 1),   # 1026, every second one block long; 2-byte aligned rows
    (32800, 33, 15, 2, 0, 2, 1),
    (21900, 25, 23, 0, 0, 2, 0),  # 1029, three a row group: in order
    (4161, 300, 9, 0, 2, 1, 2),   # 66 row groups, the last of one row
    (4161, 300, 17, 2, 0, 1, 3),
    (4224, 512, 17, 0, 0, 1, 0),  # 66 x 8 work-groups of the GEMM: in order
]


@pytest.mark.parametrize("nr,nc,nb,xpad,ypad,each,group_wgs", SIZES)
@pytest.mark.parametrize("quant", ["q4_0", "q8_0"])
def test_launch(quant, nr, nc, nb, xpad, ypad, each, group_wgs):
    (status, xs), = launches.replay([launches.gemm_call(quant, "ws", nr, nc, nb * 32, xpad, ypad)])
    assert status == 0
    assert xs[0].name == (f"pack_tiles_ranges2<{'true' if quant == 'q4_0' else 'false'}, {each}, "
                          f"{'true' if group_wgs else 'false'}>")
    groups, ranges = -(-nr // 64), -(-nb // 8)
    xgrid = -(-groups // 8) * 8 * group_wgs if group_wgs else -(-groups * ranges // each)
    assert xs[0].grid == (xgrid + -(-nc // 64) * ranges, 1, 1)


@pytest.mark.gpu
@pytest.mark.parametrize("nr,nc,nb,xpad,ypad", [s[:5] for s in SIZES])
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
