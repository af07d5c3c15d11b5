"""The x16 repack GEMM on 64- and 128-row work-groups (gemm_repack.hip) and the x4
activation pack, against the oracle bit for bit."""
import numpy as np
import pytest

import synth
from gpu_util import assert_f32_parity, from_dev, to_dev
from test_gpu_parity import x16_source

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ntok,nw,nb,bpad", [
    (4, 16, 1, 0),         # one group each way, one block
    (64, 64, 8, 0),        # one work-group, one whole chunk
    (68, 80, 24, 4),       # a second tile each way of one group; three whole chunks
    (130, 144, 21, 3),     # partial groups unwritten; two chunks and five blocks; scalar stores
    (512, 4096, 16, 0),    # 128-row work-groups, one a CU
    (516, 4112, 9, 4),     # 128-row work-groups, ragged both ways; a chunk and one block
])
def test_repack_gemm_mid(hip, oracle, dev, ntok, nw, nb, bpad):
    n = nb * 32
    w = synth.q4_0_matrix(nw, n, 501, 0.02)
    a = synth.q8_0_matrix(ntok, n, 502, 1.0)
    groups = nw // 16
    packed = oracle.pack_q4_0x16(x16_source(w[:16 * groups], nb, 18), groups * nb)
    ax4 = to_dev(np.full(ntok // 4 * nb * 136, 0xEE, np.uint8), dev)
    hip.pack_q8_0_to_q8_0x4(ntok, nb, to_dev(a, dev), a.shape[1], ax4)
    assert np.array_equal(from_dev(ax4), oracle.pack_q8_0x4(a, ntok, nb, a.shape[1]))
    bs = nw + bpad
    s = to_dev(np.full(ntok * bs, -7.0, np.float32), dev)
    hip.repack_gemm_q4_0_q8_0(n, s, to_dev(packed, dev), ax4, ntok, nw, bs)
    got = from_dev(s).reshape(ntok, bs)
    want = oracle.repack_gemm_q4_0(n, packed, from_dev(ax4), ntok, nw, bs).reshape(ntok, bs)
    rows, cols = ntok // 4 * 4, 16 * groups
    assert_f32_parity(got[:rows, :cols], want[:rows, :cols], what=f"repack {ntok}x{nw}x{n}")
    assert np.all(got[rows:] == -7.0) and np.all(got[:, cols:] == -7.0)


@pytest.mark.parametrize("bad", [0x7C00, 0xFC00, 0x7E00, 0x7BFF, 0x0001])
def test_scaled_folds_special_scales(hip, oracle, dev, bad):
    """The folds carried as 16 times the reference's (Q4_0 weights): infinite, NaN, largest
    and smallest scales on either side give the oracle's bits."""
    n, nw, ntok = 9 * 32, 48, 20
    w, a = synth.q4_0_matrix(nw, n, 503, 0.02), synth.q8_0_matrix(ntok, n, 504, 1.0)
    w.reshape(nw, 9, 18)[::5, 4, :2] = np.frombuffer(np.uint16(bad).tobytes(), np.uint8)
    a.reshape(ntok, 9, 34)[::3, 7, :2] = np.frombuffer(np.uint16(bad).tobytes(), np.uint8)
    s = to_dev(np.zeros(nw * ntok, np.float32), dev)
    hip.q4_0_q8_0_gemm(n, s, to_dev(w, dev), to_dev(a, dev), a.shape[1], nw, ntok, w.shape[1], ntok)
    want = oracle.gemm_q4_0(n, w, a, a.shape[1], nw, ntok, w.shape[1], ntok, 8)
    got = from_dev(s)
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(got[~nan].view(np.uint32), want[~nan].view(np.uint32))
    packed = oracle.pack_q4_0x16(x16_source(w, 9, 18), nw // 16 * 9)
    ax4 = oracle.pack_q8_0x4(a, ntok, 9, a.shape[1])
    hip.repack_gemm_q4_0_q8_0(n, s, to_dev(packed, dev), to_dev(ax4, dev), ntok, nw, nw)
    want = oracle.repack_gemm_q4_0(n, packed, ax4, ntok, nw, nw)
    got = from_dev(s)
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(got[~nan].view(np.uint32), want[~nan].view(np.uint32))
