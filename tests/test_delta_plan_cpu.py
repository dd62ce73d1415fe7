"""How the chunk-parallel delta rule spreads its workgroups (csrc/include/eia_delta_plan.h, as the host compiler
sees it)."""

import ctypes
import os
import shutil
import subprocess

import pytest

INCLUDE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "csrc", "include")
SOURCE = """
#include "eia_delta_plan.h"
extern "C" {
int parts(long nwg, int rep) { return dn_parts(nwg, rep); }
int first_head(int rep, int parts, int part) { return dn_first_head(rep, parts, part); }
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I", INCLUDE, str(d / "plan.cpp"), "-o",
                    str(d / "plan.so")], check=True)
    lib = ctypes.CDLL(str(d / "plan.so"))
    lib.parts.argtypes = [ctypes.c_long, ctypes.c_int]
    return lib


@pytest.mark.parametrize("rep", [1, 2, 3, 5, 8, 9, 16, 64])
def test_heads_of_a_key_head(plan, rep):
    """Every head in one part, no part empty; one head a part while there is room for it."""
    for nwg in (1, 2, 8, 31, 32, 63, 64, 65, 112, 128, 224, 256, 257, 448, 512, 513, 100000):
        n = plan.parts(nwg, rep)
        heads = [plan.first_head(rep, n, p) for p in range(n + 1)]
        assert heads[0] == 0 and heads[-1] == rep and all(b > a for a, b in zip(heads, heads[1:]))
        assert n == 1 or nwg * n <= 512
        if nwg * rep <= 512:
            assert n == rep
