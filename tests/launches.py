"""Which kernels an entry of libtcrv_hip.so launches for given arguments, without a GPU:
the library's own host code runs in a child process against tests/launch_recorder.cpp in
place of the HIP runtime, so the rules that choose a kernel are the shipped ones and not a
copy of them."""
import ctypes
import functools
import json
import os
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
LIB = os.path.join(ROOT, "tianchen-rv_amd", "libtcrv_hip.so")

# Device addresses of the replayed calls: never read, only their alignment counts.
S, X, Y, WS = 1 << 40, 2 << 40, 3 << 40, 4 << 40


class Launch:
    def __init__(self, name, grid, block):
        self.name, self.grid, self.block = name, tuple(grid), tuple(block)

    def __repr__(self):
        return f"{self.name}{self.grid}x{self.block}"


@functools.lru_cache(None)
def _recorder():
    tmp = tempfile.TemporaryDirectory()
    lib = os.path.join(tmp.name, "recorder.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-fPIC", "-shared",
                    os.path.join(HERE, "launch_recorder.cpp"), "-o", lib], check=True)
    return tmp, lib  # the folder goes with the process


def replay(calls):
    """calls: [(symbol, arguments without the stream)] -> [(status, [Launch])]."""
    out = subprocess.run([sys.executable, os.path.abspath(__file__), _recorder()[1]],
                         input=json.dumps(calls), capture_output=True, text=True)
    assert out.returncode == 0, out.stderr[-2000:]
    return [(status, [Launch(*x) for x in xs]) for status, xs in json.loads(out.stdout)]


def gemm_call(quant, entry, nr, nc, n, xpad=0, ypad=0, off=0):
    """The call of a GEMM over nr weight rows x nc tokens, operands `off` bytes past an aligned
    address and `xpad` / `ypad` bytes between rows.  entry: "plain", "ws", "tiles"
    (packed operands) or "repack" (x16 weights; nc tokens of x4 groups)."""
    nb = n // 32
    bx, by = nb * (18 if quant == "q4_0" else 34) + xpad, nb * 34 + ypad
    name = f"tcrv_hip_{quant}_q8_0_gemm"
    if entry == "plain":
        return name, (n, S, X + off, Y + off, by, nr, nc, bx, nc)
    if entry == "ws":
        return name + "_ws", (n, S, X + off, Y + off, by, nr, nc, bx, nc, WS, 1 << 50)
    if entry == "tiles":
        return name + "_tiles", (n, S, X, Y, nr, nc, nc)
    assert entry == "repack"
    return "tcrv_hip_repack_gemm_q4_0_q8_0", (n, S, X, Y, nc, nr, nr + xpad)


def kernels(calls):
    """The kernel names of each call, which has to succeed."""
    out = []
    for call, (status, xs) in zip(calls, replay(calls)):
        assert status == 0, (call, status)
        out.append([x.name for x in xs])
    return out


def main(recorder):
    sys.modules["torch"] = None  # the binding loads without it; no HIP runtime is initialised
    sys.path.insert(0, os.path.join(ROOT, "tianchen-rv_amd"))
    rec = ctypes.CDLL(recorder, mode=ctypes.RTLD_GLOBAL)
    rec.recorder_take.restype = ctypes.c_char_p
    import tcrv_hip
    out = []
    for name, args in json.load(sys.stdin):
        status = tcrv_hip.call(name, *args, 0, check=False)
        lines = rec.recorder_take().decode().splitlines()
        xs = [x.split("|") for x in lines]
        out.append((status, [(x[0], [int(v) for v in x[1:4]], [int(v) for v in x[4:]])
                             for x in xs]))
    json.dump(out, sys.stdout)


if __name__ == "__main__":
    main(sys.argv[1])
