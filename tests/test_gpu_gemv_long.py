"""The GEMV that splits long rows over a work-group's waves (gemv_long, block_dot.hip) and the
rule that takes it, through the plain entries, against the oracle bit for bit."""
import numpy as np
import pytest

import synth
from gpu_util import assert_f32_parity, assert_f32_parity_nan, from_dev, to_dev

pytestmark = pytest.mark.gpu

SHAPES = [
    # nr, nb, weight pad, output stride
    (1, 130, 0, 1),      # one row; slices of 66 and 64 blocks
    (3, 512, 0, 1),      # four whole slices, an odd row
    (767, 258, 4, 3),    # three slices of 86, padded rows, strided outputs
    (1023, 320, 0, 1),   # the last work-group half empty
    (1025, 322, 0, 1),   # Q8_0: the chunked kernel
    (2049, 160, 0, 2),   # Q8_0: two rows a work-group; Q4_0: the chunked kernel
    (4097, 192, 0, 1),   # Q8_0: two rows
    (4097, 194, 0, 1),   # Q8_0: one row
    (4096, 400, 8, 1),   # Q8_0: one row, the last 128-block chunk of 16
    (4096, 402, 0, 1),   # past it: chunked kernels
    (5, 514, 0, 1),      # past 512 blocks: chunked kernels
]


def run(hip, dev, quant, n, w, x, nr, bs):
    s = to_dev(np.full(nr * bs, -7.0, np.float32), dev)
    fn = hip.q4_0_q8_0_gemm if quant == "q4_0" else hip.q8_0_q8_0_gemm
    fn(n, s, to_dev(w, dev), to_dev(x, dev), x.shape[1], nr, 1, w.shape[1], bs)
    return from_dev(s).reshape(nr, bs)


@pytest.mark.parametrize("quant", ["q4_0", "q8_0"])
@pytest.mark.parametrize("nr,nb,pad,bs", SHAPES)
def test_gemv_long(hip, oracle, dev, quant, nr, nb, pad, bs):
    n = nb * 32
    make = synth.q4_0_matrix if quant == "q4_0" else synth.q8_0_matrix
    w = np.pad(make(nr, n, 411, 0.02), ((0, 0), (0, pad)))
    x = synth.q8_0_matrix(1, n, 412, 1.0)
    want = (oracle.gemm_q4_0 if quant == "q4_0" else oracle.gemm_q8_0)(
        n, w, x, x.shape[1], nr, 1, w.shape[1], bs, 8).reshape(nr, bs)
    got = run(hip, dev, quant, n, w, x, nr, bs)
    assert_f32_parity(got[:, :1], want[:, :1], what=f"{quant} {nr} x {n}")
    assert np.all(got[:, 1:] == -7.0)


@pytest.mark.parametrize("quant", ["q4_0", "q8_0"])
@pytest.mark.parametrize("bad", [0x7C00, 0xFC00, 0x7E00, 0x0001])
def test_gemv_long_special_scales(hip, oracle, dev, quant, bad):
    """An infinite, NaN or subnormal scale in the last block, beside the zero terms that fill
    the last 128."""
    nr, nb = 33, 258
    n = nb * 32
    size = 18 if quant == "q4_0" else 34
    w = (synth.q4_0_matrix if quant == "q4_0" else synth.q8_0_matrix)(nr, n, 413, 0.02)
    x = synth.q8_0_matrix(1, n, 414, 1.0)
    at = (nb - 1) * size
    w[::2, at], w[::2, at + 1] = bad & 0xFF, bad >> 8
    want = (oracle.gemm_q4_0 if quant == "q4_0" else oracle.gemm_q8_0)(
        n, w, x, x.shape[1], nr, 1, w.shape[1], 1, 1).reshape(nr, 1)
    got = run(hip, dev, quant, n, w, x, nr, 1)
    assert_f32_parity_nan(got, want, what=f"{quant} {bad:#x}")
