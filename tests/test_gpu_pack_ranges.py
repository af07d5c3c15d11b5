"""The GEMM-tile packs (gemm_tiled.hip; up to 128 ragged or unaligned ranges by records, the others by
8-block ranges) against the documented layout byte for
byte: the last range short by 1 to 7 blocks, rows at 2-byte alignment, one and two ranges a
work-group with an odd number of ranges, and the Q4_0 wave a range of many aligned rows."""
import numpy as np
import pytest

import synth
from gpu_util import from_dev, to_dev
from test_gpu_parity import q4_tiles_reference, tiles_reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("quant", ["q8_0", "q4_0"])
@pytest.mark.parametrize("nrows,nb,pad,off", [
    (65, 8, 0, 2),       # one range a group, two groups, the second of one row
    (64, 9, 2, 2),       # the second range stores one block of its eight
    (130, 15, 6, 14),    # and seven
    (64, 16, 4, 6),      # whole ranges off the 16-byte grid
    (6100, 65, 0, 0),    # 864 ranges: two a work-group, ragged rows of an even stride
    (6100, 72, 0, 2),    # 864 ranges, whole, 2-byte aligned
    (6100, 72, 0, 0),    # and 16-byte aligned
    (49025, 8, 0, 0),  # 767 ranges: one a work-group
    (49089, 8, 0, 0),    # 768
    (49153, 8, 0, 2),    # 769: an odd number in pairs
    (49153, 8, 0, 0),    # and in fours
])
def test_pack_ranges(hip, dev, quant, nrows, nb, pad, off):
    q4 = quant == "q4_0"
    gen = synth.q4_0_matrix if q4 else synth.q8_0_matrix
    a = np.pad(gen(nrows, nb * 32, 701, 1.0), ((0, 0), (0, pad)))
    want = (q4_tiles_reference if q4 else tiles_reference)(a, nrows, nb)
    buf = to_dev(np.zeros(a.size + 16, np.uint8), dev)
    buf[off:off + a.size] = to_dev(a.reshape(-1), dev)
    dst = to_dev(np.full(want.size + 64, 0xEE, np.uint8), dev)
    (hip.pack_q4_0_to_gemm_tiles if q4 else hip.pack_q8_0_to_gemm_tiles)(
        nrows, nb, buf[off:off + a.size], a.shape[1], dst)
    got = from_dev(dst)
    assert np.array_equal(got[:want.size], want) and np.all(got[want.size:] == 0xEE)


@pytest.mark.parametrize("quant", ["q8_0", "q4_0"])
@pytest.mark.parametrize("nr,nc,nb,pad,off", [
    (3000, 300, 11, 2, 2),  # both operands in one launch: ragged ranges, 2-byte alignment
    (3000, 300, 16, 0, 0),
])
def test_ws_pack_both(hip, oracle, dev, quant, nr, nc, nb, pad, off):
    q4, n = quant == "q4_0", nb * 32
    w = np.pad((synth.q4_0_matrix if q4 else synth.q8_0_matrix)(nr, n, 711, 0.02),
               ((0, 0), (0, pad)))
    a = np.pad(synth.q8_0_matrix(nc, n, 712, 1.0), ((0, 0), (0, pad)))
    dw, da = (to_dev(np.zeros(x.size + 16, np.uint8), dev) for x in (w, a))
    dw[off:off + w.size] = to_dev(w.reshape(-1), dev)
    da[off:off + a.size] = to_dev(a.reshape(-1), dev)
    wsb = hip.q8_0_q8_0_gemm_workspace_bytes(n, nr, nc)
    ws = to_dev(np.zeros(wsb, np.uint8), dev)
    s = to_dev(np.full(nr * nc, -7.0, np.float32), dev)
    (hip.q4_0_q8_0_gemm_ws if q4 else hip.q8_0_q8_0_gemm_ws)(
        n, s, dw[off:off + w.size], da[off:off + a.size], a.shape[1], nr, nc, w.shape[1], nc, ws,
        wsb)
    want = (oracle.gemm_q4_0 if q4 else oracle.gemm_q8_0)(
        n, w, a, a.shape[1], nr, nc, w.shape[1], nc, 16)
    assert np.array_equal(from_dev(s).view(np.uint32), want.view(np.uint32).reshape(-1))
