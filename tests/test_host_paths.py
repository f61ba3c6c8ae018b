"""Host paths that need a full device, on a stand-in for the HIP runtime (CPU
only; no kernel runs): host_paths.cpp holds the stand-in and the cases."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def host_paths(tmp_path_factory):
    from upcgen_amd import LIB_PATH
    from upcgen_amd.build import HIPCC
    exe = str(tmp_path_factory.mktemp("host_paths") / "host_paths")
    rocm = os.path.dirname(os.path.dirname(os.path.realpath(HIPCC)))
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", f"-I{rocm}/include", f"-I{ROOT}/include",
                    os.path.join(HERE, "host_paths.cpp"), "-o", exe, LIB_PATH, "-rdynamic", f"-L{rocm}/lib",
                    f"-Wl,-rpath,{os.path.dirname(LIB_PATH)}:{rocm}/lib", "-Wl,--allow-shlib-undefined"], check=True)
    return exe


@pytest.mark.parametrize("case", ["draws", "draws_full", "pairs", "pairs_full",
                                  "grid", "grid_short", "grid_full", "batch", "batch_short", "batch_full", "batch_large",
                                  "tune_shared", "tune_mixed"])
def test_host_path(host_paths, case):
    r = subprocess.run([host_paths, case], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


def test_large_draw_cases_take_the_guides(host_paths):
    from test_gpu_draw_guides_large import CASES, PART
    for nm, ny, nz, pol, n in CASES:
        for draws, want in ((n, 1), (PART, 0)):
            r = subprocess.run([host_paths, "guided"] + [str(v) for v in (nm, ny, nz, pol, draws, want)],
                               capture_output=True, text=True, timeout=60)
            assert r.returncode == 0, r.stdout + r.stderr
