"""The largest shapes the entry points take, against HIP's limit of 2^32 - 1
threads per grid axis: the host code is built as it stands and linked against a
HIP runtime that only records its launches (tests/launch_limits_check.cc).
Nothing here runs on a GPU, and no operand of these sizes is allocated."""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM", "/opt/rocm")
HIPCC = os.path.join(ROCM, "bin", "hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC) or not shutil.which("g++"), reason="hipcc or g++ not available")
def test_launches_stay_within_the_grid(tmp_path):
    inc, kdir = os.path.join(ROOT, "include"), os.path.join(ROOT, "mccl-jax_amd", "src", "kernels")
    objs, exe = [], str(tmp_path / "check")
    for src in ("reduce", "attention_bwd", "gemm", "gemm_skinny", "gemm_tiled", "attention", "attention_decode"):
        objs.append(str(tmp_path / (src + ".o")))
        subprocess.run([HIPCC, "--offload-arch=gfx950", "--cuda-host-only", "-std=c++17", "-fPIC", "-I" + inc,
                        "-I" + kdir, "-c", os.path.join(kdir, src + ".hip"), "-o", objs[-1]], check=True, timeout=300)
    # the device code's sections are left out: their registration is recorded, not read
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(ROCM, "include"), "-I" + inc,
                    os.path.join(ROOT, "tests", "launch_limits_check.cc"), *objs, "-o", exe,
                    "-Wl,--unresolved-symbols=ignore-all"], check=True, timeout=300)
    got = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert got.returncode == 0 and got.stdout.strip() == "ok", got.stdout[-2000:] + got.stderr[-2000:]
