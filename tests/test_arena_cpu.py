"""The arena of a handle's device memory (microsim_amd/csrc/gp_arena.h): a failed allocation leaves nothing behind, neither
sizes that a further try would add up, nor addresses, nor an error that the check of the next launch would find."""
import ctypes as C
import os
import subprocess

import pytest

from gp_testlib import REPO


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("arena") / "libarena.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-Wl,-Bsymbolic", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", "-I" + os.path.join(REPO, "microsim_amd", "csrc"), "-o", out,
                    os.path.join(REPO, "tests", "cpu_model", "arena_check.cpp")], check=True)
    lib = C.CDLL(out)
    lib.arena_check.argtypes, lib.arena_check.restype = [C.c_int64, C.c_int], C.c_int64
    return lib


@pytest.mark.parametrize("nbytes", [1, 256, 1000])
@pytest.mark.parametrize("tries", [1, 2, 3])
def test_retry_after_a_failed_allocation(lib, nbytes, tries):
    assert lib.arena_check(nbytes, tries) == 2 * ((nbytes + 255) // 256 * 256)
