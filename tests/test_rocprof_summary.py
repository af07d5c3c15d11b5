"""The profile summaries (tianchen-rv_amd/rocprof_summary.py) look for kernels that the library
launches for the bench's workloads, and turn counter files into bytes."""
import json
import os

import launches
import rocprof_summary


def test_kernels_are_those_of_the_workloads():
    n = 4096
    gemv = "tcrv_hip_gemv_q4_0_q8_0", (n, launches.S, launches.X, n // 32 * 18, launches.Y, n)
    calib = "tcrv_hip_add_f32", (launches.X, launches.Y, launches.S, 1 << 24)
    runs = launches.kernels([gemv, launches.gemm_call("q8_0", "plain", n, n, n),
                             launches.gemm_call("q8_0", "ws", n, n, n), calib])
    want = {"gemv_q4_0_q8_0": runs[0][0], "q8_0_q8_0_gemm": runs[1][0],
            "q8_0_q8_0_gemm_tiles": runs[2][1], "pack_both_to_gemm_tiles": runs[2][0],
            "calib": runs[3][0]}
    assert set(rocprof_summary.KERNELS) == set(want)
    for key, needle in rocprof_summary.KERNELS.items():
        assert needle in want[key], (key, needle, want[key])


def test_traffic(tmp_path, capsys):
    header = "Kernel_Name,Dispatch_Id,Counter_Value\n"
    for ctr, kib in (("FETCH_SIZE", 65536), ("WRITE_SIZE", 65536)):
        for tag, names in (("calib", ["calib"]),
                           ("gemm", ["q8_0_q8_0_gemm", "q8_0_q8_0_gemm_tiles",
                                     "pack_both_to_gemm_tiles"])):
            d = tmp_path / f"pmc_{ctr}_{tag}"
            os.makedirs(d)
            rows = [f"void tcrv::{rocprof_summary.KERNELS[name]}(...),{i},{kib}\n"
                    for i, name in enumerate(names)]
            (d / "run_counter_collection.csv").write_text(header + "".join(rows))
    rocprof_summary.traffic(str(tmp_path))
    out = json.loads(capsys.readouterr().out)
    assert out["calib_FETCH_SIZE"]["scale"] == 2.0
    # 128 MiB read (the counter reads half of it) and 64 MiB written
    assert out["pack_both_to_gemm_tiles"]["bytes"] == 192 << 20
    assert "gemv_q4_0_q8_0" not in out  # its passes were not run
