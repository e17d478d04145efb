"""The benchmark's reading of profiler output, on files as rocprofv3 writes them: it finds the
kernel that the timed apply runs, prices it as FP64 with its matrix operations, and never reports
another kernel's memory traffic for it."""
import csv
import importlib.util
import json
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
AXPY = "void pdelab_amd::axpy_kernel<double>(long long, double, double const*, double*)"


@pytest.fixture()
def bench(tmp_path, monkeypatch):
    spec = importlib.util.spec_from_file_location("bench_under_test", os.path.join(ROOT, "bench.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    monkeypatch.setattr(mod, "TRAFFIC_FILE", str(tmp_path / "traffic.json"))
    return mod


@pytest.fixture(scope="module")
def apply_name():
    """The demangled name of the library's 64^3 Q3 apply, y = J z."""
    with open(os.path.join(ROOT, "dune-pdelab_amd", "lib", "libpdelab_gpu.so"), "rb") as f:
        names = set(re.findall(rb"_ZN10pdelab_amd14dg_mfma_kernelILi4ELi0ELi0ELi0E\w+", f.read()))
    names = {subprocess.run(["c++filt"], input=n, stdout=subprocess.PIPE, check=True).stdout.decode().strip() for n in names}
    return next(n for n in names if "(" in n and "kd" not in n.split(")")[-1])


def write(path, rows):
    os.makedirs(os.path.dirname(path), exist_ok=True)
    with open(path, "w", newline="") as f:
        w = csv.DictWriter(f, list(rows[0]))
        w.writeheader()
        w.writerows(rows)


def counters(d, run, name, grid, **values):
    write(os.path.join(d, run, "x_counter_collection.csv"),
          [{"Kernel_Name": n, "Grid_Size": g, "VGPR_Count": 122, "Counter_Name": c, "Counter_Value": v}
           for n, g, vals in name_rows(name, grid, values) for c, v in vals.items()])


def name_rows(name, grid, values):
    yield name, grid, values
    if set(values) <= {"FETCH_SIZE", "WRITE_SIZE"}:
        yield AXPY, 65536, {c: 131072 for c in values}


def test_traffic_is_of_the_kernel_that_runs(bench, apply_name, tmp_path):
    d = str(tmp_path / "prof")
    write(os.path.join(d, "trace", "x_kernel_stats.csv"),
          [{"Name": apply_name, "Calls": 23, "TotalDurationNs": 1.2e6, "AverageNs": 52000.0, "Percentage": 90.0}])
    counters(d, "fetch", apply_name, 262144, FETCH_SIZE=76000)
    counters(d, "write", apply_name, 262144, WRITE_SIZE=131072)
    text = bench.profile_summary(d, 64, 3)
    # the axpy reads 16 B per DoF (2^18 KiB) and is counted as 2^17 KiB: fetched bytes count twice
    want = 76000 * 1024 * 2.0 + 131072 * 1024
    assert f"{want:.4g}" in text and bench.measured_traffic(64, 3) == pytest.approx(want)
    assert bench.measured_traffic(48, 3) is None


def test_traffic_of_another_kernel_is_not_reported(bench):
    with open(bench.TRAFFIC_FILE, "w") as f:
        json.dump({"kernel": "dg_apply_rowreg_kernel<4, double, false, false, false, false, false, false, 2>", "n": 64,
                   "degree": 3, "traffic_bytes": 1.0}, f)
    assert bench.measured_traffic(64, 3) is None


def test_counter_table_prices_the_matrix_apply(bench, apply_name, tmp_path):
    d = str(tmp_path / "prof")
    write(os.path.join(d, "trace", "x_kernel_trace.csv"),
          [{"Kernel_Name": apply_name, "Start_Timestamp": 0, "End_Timestamp": 50000}])
    n = 64 ** 3 * 64
    values = dict.fromkeys(["SQ_INSTS_VALU", "SQ_INSTS_VALU_ADD_F64", "SQ_INSTS_VALU_MUL_F64", "SQ_LDS_IDX_ACTIVE",
                            "SQ_LDS_BANK_CONFLICT", "SQ_INSTS_SALU", "SQ_INSTS_LDS", "SQ_INSTS_VMEM_RD", "SQ_INSTS_VMEM_WR",
                            "SQ_WAIT_ANY"], 0)
    values.update(GRBM_GUI_ACTIVE=8e5, SQ_WAVES=4096, SQ_WAVE_CYCLES=4e8, SQ_INSTS_VALU_FMA_F64=0.1 * 78.6e12 * 50e-6 / 128,
                  SQ_INSTS_VALU_MFMA_MOPS_F64=0.2 * 78.6e12 * 50e-6 / 512, FETCH_SIZE=8 * n / 1024 / 2, WRITE_SIZE=8 * n / 1024)
    counters(d, "pmc", apply_name, 262144, **values)
    rows = [r for r in bench.counter_summary(d).splitlines() if "dg_mfma" in r]
    assert len(rows) == 1
    cell = [c.strip() for c in rows[0].split("|")]
    # 16 B/DoF in 50 us: 0.67 of 8 TB/s; a tenth and a fifth of the FP64 rate; traffic as the algorithm's
    assert cell[2:5] == ["64^3 Q3", "50.0", "0.67"] and cell[6] == "0.30" and cell[-2] == "1.000"


def test_bytes_of_the_apply_kernels(bench):
    assert bench.apply_bytes_per_dof("dg_apply_rowreg_kernel<4, float, false, false, false, false, false, false, 2>", 3) == 8.0
    assert bench.apply_bytes_per_dof("dg_mfma_kernel<3, 3, 1, 0, 3>", 2) == 24.0
    assert bench.apply_bytes_per_dof("dg_mfma_kernel<3, 0, 0, 1, 3>", 2) == 16.0 + 8.0 * 135 / 27
    assert bench.apply_bytes_per_dof("conv_var_sq_kernel<3, float, false, true>", 2) == 12.0 + 4.0 * 135 / 27
