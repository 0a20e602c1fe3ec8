"""The library GEMM's turns (src/kernels/blas.hip): its kernels synchronise
through one workspace per GPU, so products on several streams must never
overlap, and a captured graph, which can be replayed at any time, must hold
none of them.  The host code is built as it stands and linked against a HIP
runtime and a rocBLAS that only record their calls (tests/blas_order_check.cc);
nothing here runs on a GPU."""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM", "/opt/rocm")
HIPCC = os.path.join(ROCM, "bin", "hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC) or not shutil.which("g++"), reason="hipcc or g++ not available")
def test_library_products_take_turns(tmp_path):
    inc, kdir = os.path.join(ROOT, "include"), os.path.join(ROOT, "mccl-jax_amd", "src", "kernels")
    obj, exe = str(tmp_path / "blas.o"), str(tmp_path / "check")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "--cuda-host-only", "-std=c++17", "-fPIC", "-I" + inc, "-I" + kdir,
                    "-c", os.path.join(kdir, "blas.hip"), "-o", obj], check=True, timeout=300)
    # the device code's section is left out: its registration is recorded, not read
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(ROCM, "include"), "-I" + inc,
                    os.path.join(ROOT, "tests", "blas_order_check.cc"), obj, "-o", exe, "-pthread",
                    "-Wl,--unresolved-symbols=ignore-all"], check=True, timeout=300)
    got = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert got.returncode == 0 and got.stdout.strip() == "ok", got.stdout + got.stderr
