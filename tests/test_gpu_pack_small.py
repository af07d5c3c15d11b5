"""The GEMM-tile packs on both sides of the bound between a wave a record and work-groups of
8-block ranges (gemm_tiled.hip), against the documented layout byte for byte."""
import numpy as np
import pytest

import synth
from gpu_util import from_dev, to_dev
from test_gpu_parity import q4_tiles_reference, tiles_reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("quant", ["q8_0", "q4_0"])
@pytest.mark.parametrize("nrows,nb,pad,off", [
    (1, 9, 0, 2),       # records: one row
    (4096, 9, 2, 0),    # records: 128 ranges, 2-byte aligned rows
    (4097, 9, 2, 0),    # ranges: 130, the second of a group stores one block
    (2753, 23, 0, 6),   # ranges: 132, the third stores seven; the last group has one row
    (4225, 16, 4, 14),  # ranges: 134, whole, off the 16-byte grid
])
def test_pack(hip, dev, quant, nrows, nb, pad, off):
    q4 = quant == "q4_0"
    gen = synth.q4_0_matrix if q4 else synth.q8_0_matrix
    a = np.pad(gen(nrows, nb * 32, 831, 1.0), ((0, 0), (0, pad)))
    want = (q4_tiles_reference if q4 else tiles_reference)(a, nrows, nb)
    buf = to_dev(np.concatenate([np.zeros(off, np.uint8), a.reshape(-1)]), dev)
    dst = to_dev(np.full(want.size + 64, 0xEE, np.uint8), dev)
    (hip.pack_q4_0_to_gemm_tiles if q4 else hip.pack_q8_0_to_gemm_tiles)(
        nrows, nb, buf[off:], a.shape[1], dst)
    got = from_dev(dst)
    assert np.array_equal(got[:want.size], want) and np.all(got[want.size:] == 0xEE)
