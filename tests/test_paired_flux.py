"""The flux forms of the paired-mesh kernels against the general ones, on the host."""
import os
import shutil
import subprocess

import pytest


def test_axis_fluxes_equal_the_general_forms(tmp_path):
    """Compared with == on IEEE host arithmetic: the paired kernels leave out
    terms that are exactly zero and nothing else."""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    here = os.path.dirname(os.path.abspath(__file__))
    exe = str(tmp_path / "axis_flux_check")
    subprocess.run([hipcc, "-O2", "-std=c++17", "-ffp-contract=off", "-fno-fast-math", "--offload-arch=gfx950",
                    "-I", os.path.join(here, "..", "miniaero_amd", "csrc"),
                    os.path.join(here, "host_checks", "axis_flux_check.cpp"), "-o", exe],
                   check=True, capture_output=True)
    r = subprocess.run([exe, "300000"], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
    assert r.stdout.count("mismatches=0") == 2
