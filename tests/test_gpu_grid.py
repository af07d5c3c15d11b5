"""The Q4_0 GEMM of few outputs, one wave each (block_dot_pairs over a grid), for odd block counts
and rows off the 4-byte grid: its rule, replayed without a GPU, and (-m gpu) its outputs, and
gemm_batch's just past the rule, against the oracle bit for bit."""
import numpy as np
import pytest

import launches
import synth
from gpu_util import assert_f32_parity, assert_f32_parity_nan, from_dev, to_dev

GRID = "block_dot_pairs<(DotFmt)1, false, true>"
BATCH8, BATCH16 = "gemm_batch<true, 8, false>", "gemm_batch<true, 16, false>"
ONE8, ONE16 = "gemm_batch_one<true, 8>", "gemm_batch_one<true, 16>"

SIZES = [
    # nr, nc, nb, weight pad, token pad, offset, kernel
    (1, 40, 37, 0, 0, 0, GRID),        # one weight row
    (40, 2, 9, 0, 0, 2, GRID),         # least block count
    (64, 8, 16, 2, 0, 0, GRID),        # 512 outputs
    (27, 19, 11, 0, 0, 0, BATCH8),     # 513
    (127, 8, 31, 0, 6, 0, GRID),
    (33, 31, 33, 0, 0, 0, GRID),
    (64, 32, 128, 2, 2, 0, GRID),      # one whole chunk, 2048 outputs
    (64, 33, 128, 2, 2, 0, BATCH16),   # 2112, 176 a tile
    (832, 4, 129, 0, 0, 0, GRID),      # 3328, 64 a tile
    (1665, 2, 129, 0, 0, 0, ONE8),
    (560, 5, 129, 0, 0, 0, ONE8),    # 2800, 80 a tile
    (5, 3, 257, 0, 4, 2, GRID),        # a chunk of one block
    (200, 20, 131, 0, 0, 2, BATCH8),   # three 8-wave chunks, the last of three blocks
    (1700, 2, 257, 0, 4, 0, ONE8),   # five chunks, one block in the last
    (520, 7, 65, 0, 0, 0, ONE16),    # 16 waves, nine of them with blocks
    (400, 7, 63, 2, 6, 2, ONE8),     # every slice, the last one block short
    (2, 2, 8, 2, 2, 0, ONE8),
    (4, 3, 64, 0, 0, 0, ONE8),       # 4-byte aligned rows: the rule is not for them
]


@pytest.mark.parametrize("nr,nc,nb,xpad,ypad,off,kernel", SIZES)
def test_rule(nr, nc, nb, xpad, ypad, off, kernel):
    call = launches.gemm_call("q4_0", "plain", nr, nc, nb * 32, xpad, ypad, off)
    assert launches.kernels([call]) == [[kernel]]


@pytest.mark.parametrize("nr,nc,n", [(135, 2, 11552), (1097, 2, 11936), (1, 1621, 2720),
                                      (2, 1623, 3936), (1502, 2, 9504),
                                      (517, 4, 2336)])
def test_shapes_that_gemm_batch_is_slower_at(nr, nc, n):
    assert launches.kernels([launches.gemm_call("q4_0", "plain", nr, nc, n)]) == [[GRID]]


def run(hip, dev, w, a, nr, nc, n, off):
    shifted = [to_dev(np.concatenate([np.zeros(off, np.uint8), x.reshape(-1)]), dev)[off:]
               for x in (w, a)]
    bs = nc + 3
    s = to_dev(np.full(nr * bs, -7.0, np.float32), dev)
    hip.q4_0_q8_0_gemm(n, s, *shifted, a.shape[1], nr, nc, w.shape[1], bs)
    got = from_dev(s).reshape(nr, bs)
    assert np.all(got[:, nc:] == -7.0)  # the output row padding stays untouched
    return got[:, :nc]


@pytest.mark.gpu
@pytest.mark.parametrize("nr,nc,nb,xpad,ypad,off,kernel", SIZES)
def test_parity(hip, oracle, dev, nr, nc, nb, xpad, ypad, off, kernel):
    n = nb * 32
    w = np.pad(synth.q4_0_matrix(nr, n, 811, 0.02), ((0, 0), (0, xpad)))
    a = np.pad(synth.q8_0_matrix(nc, n, 812, 1.0), ((0, 0), (0, ypad)))
    want = oracle.gemm_q4_0(n, w, a, a.shape[1], nr, nc, w.shape[1], nc, 8)
    assert_f32_parity(run(hip, dev, w, a, nr, nc, n, off), want, what=f"{kernel} {nr}x{nc}x{n}")


@pytest.mark.gpu
@pytest.mark.parametrize("bad", [0x7C00, 0xFC00, 0x7E00, 0x0001])
def test_special_scales(hip, oracle, dev, bad):
    nr, nc, nb = 33, 5, 131
    n = nb * 32
    w, a = synth.q4_0_matrix(nr, n, 813, 0.02), synth.q8_0_matrix(nc, n, 814, 1.0)
    bits = np.frombuffer(np.uint16(bad).tobytes(), np.uint8)
    w.reshape(nr, nb, 18)[::5, 130, :2] = bits
    a.reshape(nc, nb, 34)[::3, 64, :2] = bits
    want = oracle.gemm_q4_0(n, w, a, a.shape[1], nr, nc, w.shape[1], nc, 8)
    assert_f32_parity_nan(run(hip, dev, w, a, nr, nc, n, 0), want, what=f"{bad:#x}")
