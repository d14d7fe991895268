"""Addresses of the lag-window product's operand loads, on the CPU: the kernel's
own load loop compiled for the host with stand-ins for the HIP names, every
lane of every range of lags over trace lengths from one sample on, both forms
and several channels.  No load of the last row or column tile may leave
the operands' allocation."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CLANG = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "clang++")


def test_operand_loads_stay_in_the_allocation(tmp_path):
    exe = str(tmp_path / "lag_loads")
    subprocess.run([CLANG, "-O1", "-std=c++17", "-w", "-x", "c++", "-I" + os.path.join(HERE, "host", "lagstub"),
                    os.path.join(HERE, "host", "lag_loads.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
    assert r.returncode == 0, r.stdout
