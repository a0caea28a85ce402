"""The library's host code on the CPU: tests/host_path.cpp stands in for the
HIP runtime (kernels do not run), so launches that HIP would refuse, failing
allocations and failing launches can be met without a GPU."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def host_path(hip, tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("host_path") / "host_path")
    lib = os.path.join(ROOT, "hpcg_amd")
    subprocess.run(["g++", "-std=c++17", "-O1", "-rdynamic", f"-I{ROOT}/include", "-o", exe,
                    os.path.join(ROOT, "tests", "host_path.cpp"), f"-L{lib}", "-lhpcgx", f"-Wl,-rpath,{lib}",
                    "-Wl,--allow-shlib-undefined"], check=True)
    return exe


@pytest.mark.parametrize("scenario", ["one_plane", "forms_after_failure", "total_after_failure",
                                      "totals_coherent", "rz_kernels", "diagonal_after_failure"])
def test_scenario(host_path, scenario):
    out = subprocess.run([host_path, scenario], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout + out.stderr
