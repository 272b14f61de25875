"""What the HIP sources' launchers ask of the runtime, without a GPU: their host
halves compiled by hipcc and linked against a stand-in for the HIP runtime."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
HIP = os.path.join(ROOT, "jxpamg_all_amd", "csrc", "hip")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def launch(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip(f"no HIP compiler at {HIPCC}")
    d = str(tmp_path_factory.mktemp("launch"))
    objs = []
    for src in (os.path.join(HIP, "jxamd_kernels.hip"), os.path.join(HIP, "jxamd_resnorm.hip"),
                os.path.join(HERE, "hoststub", "hip_rt.cpp")):
        objs.append(os.path.join(d, os.path.basename(src) + ".o"))
        subprocess.run([HIPCC, "--offload-host-only", "-x", "hip", "--offload-arch=gfx950", "-O0", "-fPIC", "-std=c++17",
                        "-w", f"-I{ROOT}/include", f"-I{HIP}", "-c", src, "-o", objs[-1]], check=True)
    exe = os.path.join(d, "launch")
    # the device code's fat binaries are the only names left open
    subprocess.run(["g++", "-o", exe, *objs, "-Wl,--unresolved-symbols=ignore-all", "-lpthread"], check=True)
    return exe


def run(exe, what):
    r = subprocess.run([exe, what], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


def test_lds_limit_is_no_callers_own(launch):
    run(launch, "lds")


def test_residual_norm_buffers_come_back(launch):
    run(launch, "slots")
