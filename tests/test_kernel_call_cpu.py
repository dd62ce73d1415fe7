"""KernelCall passes what ctypes passes: order and width of every kind of argument, on the stack too."""

import ctypes
import random
import struct
import subprocess

import pytest

from enterprise_inference_amd import _native

TYPES = {"p": ("void*", ctypes.c_void_p), "l": ("long", ctypes.c_long), "i": ("int", ctypes.c_int),
         "f": ("float", ctypes.c_float)}
KINDS = sorted({"".join(_native._KINDS[t] for t in s) for s in _native._SIGNATURES.values()}
               | {"", "f" * 8, "i" * 64, "lf" * 8 + "p" * 48, "iiiiiiip", "ffffffff" + "i" * 9})


@pytest.fixture(scope="module")
def echo(tmp_path_factory):
    """A function per list of kinds that writes its arguments, 8 bytes each, to ``seen`` and returns -7."""
    d = tmp_path_factory.mktemp("echo")
    src = ["#include <string.h>\nunsigned char seen[64 * 8];\n"]
    for n, kinds in enumerate(KINDS):
        pars = ", ".join(f"{TYPES[k][0]} a{i}" for i, k in enumerate(kinds)) or "void"
        body = "".join(f"memcpy(seen + {8 * i}, &a{i}, sizeof a{i});" for i in range(len(kinds)))
        src.append(f"int f{n}({pars}) {{ memset(seen, 0, sizeof seen); {body} return -7; }}\n")
    (d / "echo.c").write_text("".join(src))
    subprocess.run(["gcc", "-O2", "-shared", "-fPIC", str(d / "echo.c"), "-o", str(d / "echo.so")], check=True)
    return ctypes.CDLL(str(d / "echo.so"))


def _pair(echo, n):
    fn = echo[f"f{n}"]
    fn.argtypes, fn.restype = [TYPES[k][1] for k in KINDS[n]], ctypes.c_int
    return fn, _native.runtime().KernelCall(ctypes.cast(fn, ctypes.c_void_p).value, KINDS[n], fn)


@pytest.mark.parametrize("n", range(len(KINDS)))
def test_same_arguments(echo, n):
    plain, quick = _pair(echo, n)
    seen = (ctypes.c_ubyte * 512).in_dll(echo, "seen")
    r = random.Random(n)
    pick = {"p": lambda: r.choice([None, 0, 1, r.getrandbits(47), 2 ** 64 - 8]),
            "l": lambda: r.choice([0, -1, True, r.getrandbits(62), -r.getrandbits(62)]),
            "i": lambda: r.choice([0, -1, False, 2 ** 31 - 1, -2 ** 31, r.getrandbits(30), 2 ** 32 + 5]),
            "f": lambda: r.choice([0.0, -1.5, 3, float("inf"), r.random(), 1e300])}
    for _ in range(8):
        args = [pick[k]() for k in KINDS[n]]
        assert plain(*args) == -7
        want = bytes(seen)
        assert quick(*args) == -7
        assert bytes(seen) == want, args
        for i, (k, a) in enumerate(zip(KINDS[n], args)):       # and what was meant
            if k == "i":
                assert want[8 * i:8 * i + 4] == struct.pack("<I", int(a) & 0xffffffff)
            elif k != "f":
                assert want[8 * i:8 * i + 8] == struct.pack("<Q", int(a or 0) & (2 ** 64 - 1))


def test_what_is_not_plain(echo):
    n = KINDS.index("iiiiiiip")
    plain, quick = _pair(echo, n)
    seen = (ctypes.c_ubyte * 512).in_dll(echo, "seen")
    box = ctypes.c_int(3)
    for p in (ctypes.byref(box), ctypes.c_void_p(77), (ctypes.c_long * 2)()):
        plain(*range(7), p)
        want = bytes(seen)
        quick(*range(7), p)
        assert bytes(seen) == want
    for args in ((1, 2), (*range(6), 1.5, 0), (*range(7), 2.5), (*range(6), "a", 0)):
        with pytest.raises(Exception) as a:
            plain(*args)
        with pytest.raises(type(a.value)):
            quick(*args)
    for bad in ((0, "i", plain), (1, "z", plain), (1, "f" * 9, plain), (1, "i" * 65, plain), (1, "i", 5)):
        with pytest.raises(ValueError):
            _native.runtime().KernelCall(*bad)


@pytest.mark.parametrize("sizes", [(1,), (0, 4, 0, 513), (512, 511, 1), (4096, 0), (4, 1 << 21, 5, (1 << 21) + 1, 7)])
def test_workspace_places(sizes):
    """The places of one allocation lie apart, on 512-byte steps of it, large ones on 2 MiB steps, inside it."""
    from enterprise_inference_amd.ops._dispatch import workspace
    ws, at = workspace("cpu", *sizes)
    base = ws.data_ptr()
    for a, n, b in zip(at, sizes, at[1:] + [base + ws.numel()]):
        assert (a - base) % (512 if n < 1 << 21 else 1 << 21) == 0 and a + n <= b
    assert ws.numel() >= sum(sizes)
