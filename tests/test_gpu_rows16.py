"""The short-prompt GEMM of one 16 x 16 tile a wave (gemm_rows16.hip), through the plain
and the workspace entries, against the oracle bit for bit."""
import numpy as np
import pytest

import synth
from gpu_util import assert_f32_parity, from_dev, to_dev

pytestmark = pytest.mark.gpu

SHAPES = [
    # nr, nc, nb, weight pad, token pad
    (4096, 40, 16, 0, 0),    # 256 work-groups of 32 rows and 8 tokens of a tile; one whole chunk
    (4100, 33, 17, 0, 0),    # 64-row work-groups, ragged; a chunk and one block; odd block count
    (4096, 70, 33, 2, 2),    # 32-row work-groups past two rounds; 2-byte aligned rows
    (2050, 100, 15, 0, 0),   # a partial chunk alone, odd
    (2100, 66, 34, 4, 16),   # two chunks and a pair, padded strides, 4-byte aligned rows
    (2048, 130, 1, 0, 0),    # one block
    (8200, 70, 16, 6, 0),    # rows that are not 4-byte aligned past the dword kernels' bound
]


@pytest.mark.parametrize("quant", ["q4_0", "q8_0"])
@pytest.mark.parametrize("nr,nc,nb,xpad,ypad", SHAPES)
def test_gemm_rows16(hip, oracle, dev, quant, nr, nc, nb, xpad, ypad):
    n = nb * 32
    make = synth.q4_0_matrix if quant == "q4_0" else synth.q8_0_matrix
    w = np.pad(make(nr, n, 401, 0.02), ((0, 0), (0, xpad)))
    a = np.pad(synth.q8_0_matrix(nc, n, 402, 1.0), ((0, 0), (0, ypad)))
    bs = nc + 1
    dw, da = to_dev(w, dev), to_dev(a, dev)
    want = (oracle.gemm_q4_0 if quant == "q4_0" else oracle.gemm_q8_0)(
        n, w, a, a.shape[1], nr, nc, w.shape[1], bs, 8).reshape(nr, bs)
    size = hip.q8_0_q8_0_gemm_workspace_bytes(n, nr, nc)
    ws = to_dev(np.zeros(size, np.uint8), dev)
    plain = hip.q4_0_q8_0_gemm if quant == "q4_0" else hip.q8_0_q8_0_gemm
    with_ws = hip.q4_0_q8_0_gemm_ws if quant == "q4_0" else hip.q8_0_q8_0_gemm_ws
    for run, extra in ((plain, ()), (with_ws, (ws, size))):
        s = to_dev(np.full(nr * bs, -7.0, np.float32), dev)
        run(n, s, dw, da, a.shape[1], nr, nc, w.shape[1], bs, *extra)
        got = from_dev(s).reshape(nr, bs)
        assert_f32_parity(got[:, :nc], want[:, :nc], what=f"{quant} {nr}x{nc}x{n}")
        assert np.all(got[:, nc:] == -7.0)
