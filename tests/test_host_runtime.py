"""Host code of the engine over a stand-in HIP runtime in host memory
(fake_hip.cpp; kernels are not run): buffers kept by a context, the host copies
it makes, several threads, calls that fail on the way."""
import subprocess
from pathlib import Path

import pytest

from proteindf_amd import engine

ROOT = Path(__file__).resolve().parents[1]
TESTS = ROOT / "tests"


@pytest.fixture(scope="session")
def program(tmp_path_factory):
    """host_checks.cpp (signed overflow ends it) linked to the stand-in first, the engine library second."""
    out = tmp_path_factory.mktemp("host")
    cxx = ["g++", "-std=c++17", "-O1", "-g", "-ftrapv", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", f"-I{ROOT / 'include'}",
           f"-I{ROOT / 'proteindf_amd' / 'csrc'}"]
    fake, lib = out / "libfake.so", Path(engine.LIB_PATH)
    subprocess.run(cxx + ["-fPIC", "-shared", str(TESTS / "fake_hip.cpp"), "-o", str(fake)], check=True)
    subprocess.run(cxx + [str(TESTS / "host_checks.cpp"), "-o", str(out / "checks"), str(fake), str(lib), "-pthread",
                          f"-Wl,-rpath,{out},-rpath,{lib.parent}", "-Wl,--allow-shlib-undefined"], check=True)
    return out / "checks"


@pytest.mark.parametrize("check", ["pool_threads", "host_copy_threads", "grid_rows", "pool_bound",
                                   "reserve_gives_way", "density_keeps_little", "failed_copies", "part_tree_sizes",
                                   "rho_without_memory", "small_grids"])
def test_host_code(program, check):
    r = subprocess.run([str(program), check], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
