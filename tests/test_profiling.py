"""The reducer of rocprofv3 output (profiling.py) on made-up CSV files of the
profiler's columns: the read counter is calibrated on the conversion kernels, and
a run without one is refused, not scaled by a constant."""
import csv

import pytest

from lowmachmixtures_amd import profiling

MARCH = "void lmm::(anonymous namespace)::k_rb_march2x3<float, lmm::StagRB<float, 0, -1>, lmm::StagRB<float, 1, -1>, " \
        "lmm::StagRB<float, 2, -1>, 64, false, 2>(Grid)"


def _write(path, cols, rows):
    path.parent.mkdir(parents=True)
    with open(path, "w", newline="") as f:
        w = csv.writer(f)
        w.writerow(cols)
        w.writerows(rows)


def _run(tmp_path, convert, n=256):
    N = n ** 3
    kernels = [(convert, 8 * N, 8 * 8 * N, 4 * 8 * N), (MARCH, N, 60 * N, 12 * N)]  # name, work-items, read, written
    _write(tmp_path / "trace" / "run_kernel_trace.csv",
           ["Kernel_Name", "Dispatch_Id", "Start_Timestamp", "End_Timestamp", "Grid_Size_X"],
           [[k[0], i + 1, 1000 * i, 1000 * i + 500, k[1]] for i, k in enumerate(kernels)])
    # the counter sees half of every read
    for d, counter, q, scale in (("pmc_f", "FETCH_SIZE", 2, 0.5), ("pmc_w", "WRITE_SIZE", 3, 1.0)):
        _write(tmp_path / d / "run_counter_collection.csv",
               ["Dispatch_Id", "Kernel_Name", "Grid_Size", "Counter_Name", "Counter_Value"],
               [[i + 1, k[0], k[1], counter, k[q] * scale / 1024] for i, k in enumerate(kernels)])
    out = tmp_path / "trace.txt", tmp_path / "counters.txt"
    profiling.summarize(str(tmp_path), n, "bench", str(out[0]), str(out[1]))
    return out[1].read_text()


def test_calibrated_on_the_conversion_list(tmp_path):
    text = _run(tmp_path, "lmm::k_convert_list(lmm::ConvertList, long)")
    assert "true read / FETCH_SIZE = 2.000 (median of 1 dispatches" in text
    assert f"traffic fp32_mg 256 {72 * 256 ** 3}" in text


def test_no_calibration_is_an_error(tmp_path):
    with pytest.raises(ValueError, match="calibrate"):
        _run(tmp_path, "lmm::k_fill<double>(double*, long, double)")
