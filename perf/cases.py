"""Workloads of the quantized kernels as a program that serves a ggml-quantized
model calls them through the Python binding (tianchen-rv_amd/tcrv_hip.py): decode
GEMVs, batched decode, prompts, prefill, and the row codecs, over the sizes of
bench.py and the tests.

A case is a dict of plain values:
  kind    "gemv" | "gemm" | "codec"
  quant   "q4_0" | "q8_0": the weights' format (activations are Q8_0)
  entry   how the weights are kept and which entry runs them:
            gemv:  "plain" rows, "x16" repacked groups, "soa" split planes (Q4_0)
            gemm:  "plain" rows, "ws" plain rows with a caller's workspace,
                   "tiles" weights packed once and activations packed per call,
                   "repack" x16 weights (Q4_0), activations interleaved per call
            codec: "rows"
  n       the contraction length K (codec: the row length), a multiple of 32
  nr      weight rows (codec: rows)
  nc      tokens (gemm)

listed() are the fixed cases, draw(rng) gives another of the same ranges,
prepare(case, seed) makes the device buffers, run(state) is one pass, work(case)
the bytes and operations that no implementation can do without, exact(case, seed)
the results in float64 by plain torch.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "tianchen-rv_amd"))
import tcrv_hip  # noqa: E402

QK = 32
BLOCK_BYTES = {"q4_0": 18, "q8_0": 34}
DEV = "cuda:0"

# The ranges that draw() spreads over; the listed cases lie inside them.
N_RANGE = (1024, 14336)
GEMV_ROWS = (512, 32000)
GEMM_ROWS = (512, 14336)
CODEC_ROWS = (64, 4096)
MOST_WEIGHTS = 32000 * 4096          # weights of a GEMV
MOST_MACS = 4096 ** 3                # of a GEMM


def listed():
    return [
        # The smallest call: one projection of a small model for one token; launch and latency.
        dict(name="gemv_q4_small", kind="gemv", quant="q4_0", entry="plain", n=1024, nr=1024),
        # The output head of a 32000-word vocabulary for one token: the largest decode read.
        dict(name="gemv_q4_head", kind="gemv", quant="q4_0", entry="plain", n=4096, nr=32000),
        # The feed-forward down projection for one token with Q8_0 weights: long rows.
        dict(name="gemv_q8_down", kind="gemv", quant="q8_0", entry="plain", n=14336, nr=4096),
        # The feed-forward up projection for one token over x16-repacked weights.
        dict(name="gemv_x16_up", kind="gemv", quant="q4_0", entry="x16", n=4096, nr=14336),
        # Batched decode: sixteen sequences' next tokens through one projection.
        dict(name="batch_q8_16", kind="gemm", quant="q8_0", entry="plain", n=4096, nr=4096, nc=16),
        # Batched decode with ragged sizes: an odd block count (rows only 2-byte aligned), six
        # sequences, weight rows that fill no tile.
        dict(name="batch_q4_odd", kind="gemm", quant="q4_0", entry="plain", n=2912, nr=3001, nc=6),
        # A short prompt (or many sequences' decode) through one projection, plain rows.
        dict(name="prompt_q4_128", kind="gemm", quant="q4_0", entry="plain", n=4096, nr=4096,
             nc=128),
        # A prompt with ragged sizes and an odd block count, through the workspace entry.
        dict(name="prompt_q8_odd", kind="gemm", quant="q8_0", entry="ws", n=2912, nr=3001, nc=333),
        # Prefill of a long prompt, plain rows with a workspace: the largest product.
        dict(name="prefill_q8_ws", kind="gemm", quant="q8_0", entry="ws", n=4096, nr=4096,
             nc=4096),
        # Prefill over weights packed at load time, a prompt of no round length.
        dict(name="prefill_q4_tiles", kind="gemm", quant="q4_0", entry="tiles", n=4096, nr=11008,
             nc=1000),
        # A prompt over x16-repacked weights, its activations interleaved first.
        dict(name="prompt_x16_512", kind="gemm", quant="q4_0", entry="repack", n=4096, nr=4096,
             nc=512),
        # The codecs over one projection's size: activations quantized, weights expanded.
        dict(name="codec_q8", kind="codec", quant="q8_0", entry="rows", n=4096, nr=4096),
    ]


def _log_uniform(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(("gemv", "gemv", "batch", "batch", "prompt", "prompt", "prefill", "codec"))
    quant = rng.choice(("q4_0", "q8_0"))
    # Half of the models have rows of whole 256s, the others any multiple of a block.
    n = _log_uniform(rng, *N_RANGE)
    n = n // 256 * 256 if rng.random() < 0.5 else n // QK * QK
    if kind == "codec":
        return dict(kind="codec", quant=quant, entry="rows", n=min(n, 4096),
                    nr=_log_uniform(rng, *CODEC_ROWS))
    if kind == "gemv":
        entry = rng.choice(("plain", "plain", "x16", "soa") if quant == "q4_0" else
                           ("plain", "plain", "x16"))
        nr = min(_log_uniform(rng, *GEMV_ROWS), MOST_WEIGHTS // n)
        if entry == "x16":
            nr = nr // 16 * 16
        if entry == "soa":
            n = n // 64 * 64
        return dict(kind="gemv", quant=quant, entry=entry, n=n, nr=nr)
    if kind == "batch":
        entry, nc = "plain", _log_uniform(rng, 2, 64)
    elif kind == "prompt":
        entry, nc = rng.choice(("plain", "ws", "tiles", "repack")), _log_uniform(rng, 65, 512)
    else:
        entry, nc = rng.choice(("ws", "tiles", "repack")), _log_uniform(rng, 513, 4096)
    nr = _log_uniform(rng, *GEMM_ROWS)
    if entry == "repack":
        quant, nc, nr = "q4_0", nc // 4 * 4, nr // 16 * 16
    nr = min(nr, MOST_MACS // (n * nc) // 16 * 16)
    return dict(kind="gemm", quant=quant, entry=entry, n=n, nr=nr, nc=nc)


# ---------------------------------------------------------------------------
# Inputs: normal weights (std 0.02) and activations (std 1), quantized as ggml
# quantizes them, on the device.
# ---------------------------------------------------------------------------

def _normal(gen, rows, n, std):
    return torch.randn(rows, n, generator=gen, device=DEV, dtype=torch.float32) * std


def _scaled(x, d):
    """x / d per block, with 0 where d is 0 (as x times ggml's guarded reciprocal)."""
    return x * torch.where(d == 0, torch.zeros_like(d), 1.0 / d)[..., None]


def _bytes_of_halves(d):
    return d.half().contiguous().view(torch.uint8).reshape(*d.shape, 2)


def _quantize(quant, x):
    """float32 [rows, n] -> uint8 [rows, n / 32 * block bytes]."""
    rows, n = x.shape
    xb = x.reshape(rows, n // QK, QK)
    amax, at = xb.abs().max(dim=-1)
    if quant == "q8_0":
        d = amax / 127.0
        q = _scaled(xb, d).round().clamp(-127, 127).to(torch.int8).view(torch.uint8)
    else:
        d = xb.gather(-1, at[..., None])[..., 0] / -8.0
        q = (_scaled(xb, d) + 8.5).floor().clamp(0, 15).to(torch.uint8)
        q = q[..., :16] | (q[..., 16:] << 4)
    return torch.cat([_bytes_of_halves(d), q], dim=-1).reshape(rows, -1).contiguous()


def _values(quant, rows):
    """float64 values of quantized rows (uint8 [rows, bytes])."""
    b = rows.reshape(rows.shape[0], -1, BLOCK_BYTES[quant])
    d = b[..., :2].contiguous().view(torch.float16).double()
    q = b[..., 2:].contiguous()
    if quant == "q8_0":
        v = q.view(torch.int8).double()
    else:
        v = torch.cat([(q & 15).double(), (q >> 4).double()], dim=-1) - 8.0
    return (v * d).reshape(rows.shape[0], -1)


def _inputs(case, seed):
    """(weights, activations): quantized rows; the codec's activations are float32."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    w = _quantize(case["quant"], _normal(gen, case["nr"], case["n"], 0.02))
    tokens = case["nr"] if case["kind"] == "codec" else case.get("nc", 1)
    a = _normal(gen, tokens, case["n"], 1.0)
    return w, a if case["kind"] == "codec" else _quantize("q8_0", a)


def _buffer(nbytes):
    return torch.empty(nbytes, dtype=torch.uint8, device=DEV)


def _x16(quant, w, nb):
    """Plain rows -> x16 groups: block b of 16 consecutive rows interleaved."""
    nr, bb = w.shape[0], BLOCK_BYTES[quant]
    src = w.reshape(nr // 16, 16, nb, bb).transpose(1, 2).contiguous()
    dst = _buffer(nr * nb * bb)
    pack = tcrv_hip.pack_q4_0_to_q4_0x16 if quant == "q4_0" else tcrv_hip.pack_q8_0_to_q8_0x16
    pack(nr // 16 * nb, src, dst)
    return dst


def prepare(case, seed):
    """The device buffers of a case and the calls of one pass over them: {"calls": [(entry,
    arguments)], "out": what a pass computes}."""
    kind, quant, entry, n, nr = (case[k] for k in ("kind", "quant", "entry", "n", "nr"))
    nb = n // QK
    w, a = _inputs(case, seed)
    bx, by = w.shape[1], a.shape[1]
    if kind == "codec":
        packed = _buffer(nr * nb * 34)
        wide = torch.empty(nr, n, dtype=torch.float32, device=DEV)
        expand = (tcrv_hip.dequantize_row_q4_0 if quant == "q4_0" else
                  tcrv_hip.dequantize_row_q8_0)
        return {"calls": [(tcrv_hip.quantize_row_q8_0, (nr * n, a, packed)),
                          (expand, (w, wide, nr * n))],
                "out": {"quantized": packed, "expanded": wide}}
    if kind == "gemv":
        s = torch.empty(nr, dtype=torch.float32, device=DEV)
        if entry == "x16":
            fn = (tcrv_hip.repack_gemv_q4_0_q8_0 if quant == "q4_0" else
                  tcrv_hip.repack_gemv_q8_0_q8_0)
            call = (fn, (n, s, _x16(quant, w, nb), a, nr))
        elif entry == "soa":
            soa = _buffer(nr * nb * 18)
            tcrv_hip.pack_q4_0_to_soa(nr, nb, w, bx, soa)
            call = (tcrv_hip.gemv_q4_0_soa_q8_0, (n, s, soa, a, nr))
        elif quant == "q4_0":
            call = (tcrv_hip.gemv_q4_0_q8_0, (n, s, w, bx, a, nr))
        else:
            call = (tcrv_hip.q8_0_q8_0_gemm, (n, s, w, a, by, nr, 1, bx, 1))
        return {"calls": [call], "out": s}
    nc = case["nc"]
    if entry == "repack":
        s = torch.empty(nc, nr, dtype=torch.float32, device=DEV)
        a4 = _buffer(nc * nb * 34)
        return {"calls": [(tcrv_hip.pack_q8_0_to_q8_0x4, (nc, nb, a, by, a4)),
                          (tcrv_hip.repack_gemm_q4_0_q8_0,
                           (n, s, _x16(quant, w, nb), a4, nc, nr, nr))],
                "out": s}
    s = torch.empty(nr, nc, dtype=torch.float32, device=DEV)
    q4 = quant == "q4_0"
    if entry == "plain":
        fn = tcrv_hip.q4_0_q8_0_gemm if q4 else tcrv_hip.q8_0_q8_0_gemm
        calls = [(fn, (n, s, w, a, by, nr, nc, bx, nc))]
    elif entry == "ws":
        size = (tcrv_hip.q4_0_q8_0_gemm_workspace_bytes if q4 else
                tcrv_hip.q8_0_q8_0_gemm_workspace_bytes)(n, nr, nc)
        fn = tcrv_hip.q4_0_q8_0_gemm_ws if q4 else tcrv_hip.q8_0_q8_0_gemm_ws
        calls = [(fn, (n, s, w, a, by, nr, nc, bx, nc, _buffer(size), size))]
    else:
        tx = _buffer(tcrv_hip.gemm_tiles_bytes(nr, nb))
        ty = _buffer(tcrv_hip.gemm_tiles_bytes(nc, nb))
        pack = tcrv_hip.pack_q4_0_to_gemm_tiles if q4 else tcrv_hip.pack_q8_0_to_gemm_tiles
        pack(nr, nb, w, bx, tx)
        fn = tcrv_hip.q4_0_q8_0_gemm_tiles if q4 else tcrv_hip.q8_0_q8_0_gemm_tiles
        calls = [(tcrv_hip.pack_q8_0_to_gemm_tiles, (nc, nb, a, by, ty)),
                 (fn, (n, s, tx, ty, nr, nc, nc))]
    return {"calls": calls, "out": s}


def run(state):
    for entry, arguments in state["calls"]:
        entry(*arguments)
    return state["out"]


def work(case):
    n, nr, nc = case["n"], case["nr"], case.get("nc", 1)
    w = nr * n // QK * BLOCK_BYTES[case["quant"]]
    if case["kind"] == "codec":
        return {"bytes": nr * n * 4 + nr * n // QK * 34 + w + nr * n * 4, "flops": 2 * nr * n}
    return {"bytes": w + nc * n // QK * 34 + nr * nc * 4, "flops": 2 * nr * nc * n}


def tolerance(case):
    """The entries promise the reference's fold, one rounding after another in ascending block
    order, so every output is the same bit for bit whichever kernel computes it."""
    return "exact"


def exact(case, seed):
    w, a = _inputs(case, seed)
    wide = _values(case["quant"], w)
    if case["kind"] == "codec":
        return {"quantized": None, "expanded": wide}
    if case["kind"] == "gemv":
        return (wide @ _values("q8_0", a)[0]).contiguous()
    y = _values("q8_0", a)
    return y @ wide.t() if case["entry"] == "repack" else wide @ y.t()
