"""Host-side checks of the LDS GEMM's plan, compiled from
tests/native/gemm_plan_check.cpp against the built library: tiles and k-splits
for every ESM-2 projection when the caller has all, some or none of the room
for partial sums that the splits want."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(os.path.dirname(HERE), "codon-infer_amd", "codon_hip")


def test_plan_fits_the_room_for_partial_sums(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc) or not os.path.exists(os.path.join(LIB, "libcodon_hip.so")):
        pytest.skip("hipcc or the built library not available")
    exe = str(tmp_path / "gemm_plan_check")
    src = os.path.join(HERE, "native", "gemm_plan_check.cpp")
    r = subprocess.run([hipcc, "-O1", "-std=c++17", "-Wno-unused-result", "-x", "hip", "--offload-arch=gfx950", "-o",
                        exe, src, "-x", "none", "-L" + LIB, "-lcodon_hip", "-Wl,-rpath," + LIB],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    env = {k: v for k, v in os.environ.items() if not k.startswith("CIH_")}
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60, env=env)
    print(out.stdout)
    assert out.returncode == 0 and out.stdout.strip().endswith("OK"), out.stdout[-2000:]
