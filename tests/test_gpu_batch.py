"""The 16 x 16-tile GEMM that splits K over a work-group's waves (gemm_batch.hip),
through the plain GEMM, GEMV and workspace entries, against the oracle bit for bit:
few tokens, and rows that are only 2-byte aligned at any number of tokens (Q4_0 runs a few of
these sizes a wave an output; its own past that rule are in test_gpu_grid.py)."""
import numpy as np
import pytest
import torch

import synth
from gpu_util import assert_f32_parity, empty_dev, from_dev, to_dev

pytestmark = pytest.mark.gpu


def matrix(quant, rows, n, seed, std):
    return (synth.q4_0_matrix if quant == "q4_0" else synth.q8_0_matrix)(rows, n, seed, std)


def shifted(a, off, dev):
    """The bytes of `a` on the device, `off` bytes past an aligned address."""
    return to_dev(np.concatenate([np.zeros(off, np.uint8), a.reshape(-1)]), dev)[off:]


SHAPES = [
    # nr, nc, nb, weight pad, token pad, offset
    (16, 5, 1, 0, 0, 0),       # one block: a partial slice of 18 / 34 bytes
    (17, 16, 8, 0, 0, 0),      # one whole slice; a second tile of one row
    (40, 17, 9, 0, 0, 0),      # odd block count (2-byte aligned rows); a second token group
    (33, 7, 63, 2, 6, 2),      # every slice of an 8-wave chunk, the last one block short
    (130, 3, 64, 0, 0, 0),     # exactly one 8-wave chunk, three tokens
    (21, 6, 65, 0, 0, 0),      # 16 waves, nine of them with blocks
    (4096, 16, 128, 0, 0, 0),  # 16 waves, one whole chunk, a work-group a CU
    (48, 33, 128, 2, 2, 0),    # 2-byte aligned rows, three token groups, whole chunk
    (37, 20, 131, 0, 0, 2),    # three 8-wave chunks, the last of three blocks
    (20, 2, 257, 0, 4, 0),     # five chunks, one block in the last
    (300, 70, 11, 0, 0, 0),    # unaligned rows past 64 tokens
    (4100, 1, 91, 0, 0, 0),    # decode over odd rows
    (1, 40, 37, 0, 0, 0),      # one weight row, odd block count
    (1, 1, 3, 0, 0, 2),        # one output
]


@pytest.mark.parametrize("quant", ["q4_0", "q8_0"])
@pytest.mark.parametrize("nr,nc,nb,xpad,ypad,off", SHAPES)
def test_gemm_batch(hip, oracle, dev, quant, nr, nc, nb, xpad, ypad, off):
    n = nb * 32
    w = np.pad(matrix(quant, nr, n, 301, 0.02), ((0, 0), (0, xpad)))
    a = np.pad(matrix("q8_0", nc, n, 302, 1.0), ((0, 0), (0, ypad)))
    bs = nc + 3
    s = to_dev(np.full(nr * bs, -7.0, np.float32), dev)
    run = hip.q4_0_q8_0_gemm if quant == "q4_0" else hip.q8_0_q8_0_gemm
    run(n, s, shifted(w, off, dev), shifted(a, off, dev), a.shape[1], nr, nc, w.shape[1], bs)
    want = (oracle.gemm_q4_0 if quant == "q4_0" else oracle.gemm_q8_0)(
        n, w, a, a.shape[1], nr, nc, w.shape[1], bs, 8).reshape(nr, bs)
    got = from_dev(s).reshape(nr, bs)
    assert_f32_parity(got[:, :nc], want[:, :nc], what=f"{quant} {nr}x{nc}x{n}")
    assert np.all(got[:, nc:] == -7.0)  # the output row padding stays untouched


@pytest.mark.parametrize("quant", ["q4_0", "q8_0"])
def test_gemm_batch_strides_past_256_mb(hip, oracle, dev, quant):
    """Row strides past the kernel's 32-bit row offsets (64-bit ones there)."""
    nr, nc, nb, stride = 3, 2, 5, (1 << 28) + 6
    n = nb * 32
    w, a = matrix(quant, nr, n, 303, 0.02), matrix("q8_0", nc, n, 304, 1.0)
    dw = torch.zeros(2 * stride + w.shape[1], dtype=torch.uint8, device=dev)
    da = torch.zeros(stride + a.shape[1], dtype=torch.uint8, device=dev)
    for rows, buf in ((w, dw), (a, da)):
        for r, row in enumerate(rows):
            buf[r * stride:r * stride + row.size] = torch.from_numpy(row).to(dev)
    s = empty_dev(nr * nc, torch.float32, dev)
    run = hip.q4_0_q8_0_gemm if quant == "q4_0" else hip.q8_0_q8_0_gemm
    run(n, s, dw, da, stride, nr, nc, stride, nc)
    want = (oracle.gemm_q4_0 if quant == "q4_0" else oracle.gemm_q8_0)(
        n, w, a, a.shape[1], nr, nc, w.shape[1], nc, 8)
    assert_f32_parity(from_dev(s), want, what=f"{quant} wide strides")


@pytest.mark.parametrize("quant", ["q4_0", "q8_0"])
def test_gemm_ws_few_tokens_checks_its_workspace(hip, oracle, dev, quant):
    """Few tokens through the workspace entries run on the plain rows: the workspace is
    left untouched, and a missing or short one is still refused."""
    nr, nc, nb = 272, 40, 9
    n = nb * 32
    w, a = matrix(quant, nr, n, 305, 0.02), matrix("q8_0", nc, n, 306, 1.0)
    dw, da = to_dev(w, dev), to_dev(a, dev)
    s = empty_dev(nr * nc, torch.float32, dev)
    size = (hip.q4_0_q8_0_gemm_workspace_bytes if quant == "q4_0" else
            hip.q8_0_q8_0_gemm_workspace_bytes)(n, nr, nc)
    run = hip.q4_0_q8_0_gemm_ws if quant == "q4_0" else hip.q8_0_q8_0_gemm_ws
    ws = torch.full((size,), 0xA5, dtype=torch.uint8, device=dev)
    for bad, nbytes, status in ((None, size, hip.ERR_NULL_POINTER), (ws, size - 1, hip.ERR_BAD_SIZE)):
        with pytest.raises(hip.TcrvHipError) as e:
            run(n, s, dw, da, a.shape[1], nr, nc, w.shape[1], nc, bad, nbytes)
        assert e.value.status == status
    run(n, s, dw, da, a.shape[1], nr, nc, w.shape[1], nc, ws, size)
    want = (oracle.gemm_q4_0 if quant == "q4_0" else oracle.gemm_q8_0)(
        n, w, a, a.shape[1], nr, nc, w.shape[1], nc, 8)
    assert_f32_parity(from_dev(s), want, what=f"{quant} ws {nr}x{nc}x{n}")
    assert bool(torch.all(ws == 0xA5))
