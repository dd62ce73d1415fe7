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
int xcds(int G, int per_kv) { return 1 << dn_spread(G, per_kv).shift; }
int grid(int G, int per_kv, int nseq) { return dn_grid(nseq * G, dn_spread(G, per_kv)); }
int place(int block, int G, int per_kv, int* kv) {
  const DeltaWg wg = dn_place(block, dn_spread(G, per_kv));
  *kv = wg.kv;
  return wg.in;
}
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


@pytest.mark.parametrize("per_kv", [1, 2, 3, 8, 15, 16, 32, 64, 128])
@pytest.mark.parametrize("G", [1, 2, 3, 4, 5, 6, 7, 8, 9, 12, 16, 24])
@pytest.mark.parametrize("nseq", [1, 2, 3, 7])
def test_workgroups_of_the_scan(plan, nseq, G, per_kv):
    """Every (sequence, key head) and column group once; and all XCDs take the same share of every sequence."""
    x, kvs = plan.xcds(G, per_kv), nseq * G
    kv, seen, full = ctypes.c_int(), set(), [0] * 8
    for b in range(plan.grid(G, per_kv, nseq)):
        at = plan.place(b, G, per_kv, ctypes.byref(kv))
        if kv.value < kvs and at < per_kv:
            assert at >= 0 and (kv.value, at) not in seen
            seen.add((kv.value, at))
            full[b % 8] += 1
    assert len(seen) == kvs * per_kv and x == (1 if G % 8 == 0 else 8 // G if 8 % G == 0 else 2)
    if (G % 8 == 0 or 8 % G == 0) and per_kv % x == 0:
        assert max(full) == min(full) == kvs * per_kv // 8
    assert max(full) <= -(-kvs * x // 8) * -(-per_kv // x)
