"""Parts of the lag-window kernel on the CPU, compiled for the host with stand-ins
for the HIP names.

Addresses of the product's operand loads: every lane of every range of lags over
trace lengths from one sample on, both forms and several channels.  No load of the last row or column tile may leave
the operands' allocation.

The scan's running state among values that differ in their last bits."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CLANG = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "clang++")


def _run(tmp_path, program):
    exe = str(tmp_path / "program")
    subprocess.run([CLANG, "-O1", "-std=c++17", "-w", "-x", "c++", "-I" + os.path.join(HERE, "host", "lagstub"),
                    os.path.join(HERE, "host", program), "-o", exe], check=True)
    r = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
    assert r.returncode == 0, r.stdout


def test_operand_loads_stay_in_the_allocation(tmp_path):
    _run(tmp_path, "lag_loads.cpp")


def test_scan_state(tmp_path):
    _run(tmp_path, "lag_scan.cpp")


def test_tile_kernel_loads_stay_in_the_planes(tmp_path):
    _run(tmp_path, "lag_tile_loads.cpp")
