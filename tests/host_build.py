"""Compiles a program of tests/host against the engine's host sources with the
stand-in of the HIP runtime (tests/host/standin.h) and runs it."""
import os
import subprocess
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
HOST = os.path.join(HERE, "host")
CSRC = os.path.join(os.path.dirname(HERE), "seismic_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
CLANG = os.path.join(ROCM, "llvm", "bin", "clang++")


def run_host(tmp_path, program, sources, *args):
    """Builds HOST/program with the named engine sources and runs it with args;
    returns (status, output)."""
    srcs = [os.path.join(HOST, program), os.path.join(HOST, "standin.cpp")] + [os.path.join(CSRC, s) for s in sources]
    objs = [str(tmp_path / (os.path.basename(s) + ".o")) for s in srcs]

    def compile_one(so):
        subprocess.run([CLANG, "-O1", "-g", "-std=c++17", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}/include", "-w", "-c", so[0],
                        "-o", so[1]], check=True)

    with ThreadPoolExecutor(4) as pool:
        list(pool.map(compile_one, zip(srcs, objs)))
    exe = str(tmp_path / "program")
    subprocess.run([CLANG, *objs, "-lpthread", "-o", exe], check=True)
    r = subprocess.run([exe, *args], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    return r.returncode, r.stdout
