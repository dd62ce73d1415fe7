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
void solve(int G, int nchunk, int rep, long* out) {
  const DeltaSolve s = dn_solve(G, nchunk, rep);
  out[0] = s.whole; out[1] = s.parts; out[2] = s.blocks;
}
void solve_place(long block, int G, int whole, int parts, int* out) {
  const DeltaSolveWg w = dn_solve_place(block, G, whole, parts);
  out[0] = w.chunk; out[1] = w.kh; out[2] = w.parts; out[3] = w.part;
}
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


@pytest.mark.parametrize("rep", [1, 2, 3, 8])
@pytest.mark.parametrize("G", [1, 3, 7, 8, 16, 513])
@pytest.mark.parametrize("nchunk", [1, 2, 63, 64, 65, 66, 170, 171, 172, 300])
def test_workgroups_of_the_solve(plan, nchunk, G, rep):
    """Every head of every chunk once; heads are spread in the last round of 512 workgroups only."""
    out, wg = (ctypes.c_long * 3)(), (ctypes.c_int * 4)()
    plan.solve(G, nchunk, rep, out)
    whole, parts, blocks = out
    assert 0 <= whole <= nchunk and whole * G <= G * nchunk // 512 * 512
    assert G * (nchunk - whole) * parts <= 512 or parts == 1
    plan.solve_place.argtypes = [ctypes.c_long, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_void_p]
    heads = set()
    for b in range(blocks):
        plan.solve_place(b, G, whole, parts, wg)
        chunk, kh, n, part = wg
        assert 0 <= chunk < nchunk and 0 <= kh < G and 0 <= part < n
        mine = {(chunk, kh, h) for h in range(plan.first_head(rep, n, part), plan.first_head(rep, n, part + 1))}
        assert mine and not mine & heads
        heads |= mine
    assert len(heads) == nchunk * G * rep


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
