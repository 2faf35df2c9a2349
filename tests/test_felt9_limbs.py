"""The nine-limb products and the partial round of the device Poseidon (stwo-ml_amd/csrc/felt9.h,
poseidon9.h), built for the CPU, at the largest limbs and values their comments allow: every 64-bit
column and 32-bit carry has to hold there.  Checked against Python integers."""
import ctypes as C
import os
import random
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "tests", "native", "felt9_limbs.cpp")
OUT = os.path.join(ROOT, "tests", "native", "_build", "libfelt9_limbs.so")
CLANG = "/opt/rocm/llvm/bin/clang++"
PF = (1 << 251) + 17 * (1 << 192) + 1
R = 1 << 261
M29 = (1 << 29) - 1


@pytest.fixture(scope="module")
def f9():
    deps = [SRC] + [os.path.join(ROOT, "stwo-ml_amd", "csrc", f) for f in
                    ("felt9.h", "poseidon9.h", "poseidon9_host.h", "poseidon.h", "felt252.h")]
    if not os.path.exists(OUT) or os.path.getmtime(OUT) < max(os.path.getmtime(d) for d in deps):
        if not os.path.exists(CLANG):
            pytest.skip("clang++ from ROCm not available")
        os.makedirs(os.path.dirname(OUT), exist_ok=True)
        subprocess.run([CLANG, "-O2", "-std=c++17", "-mbmi2", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                        "-I/opt/rocm/include", "-o", OUT, SRC], check=True)
    return C.CDLL(OUT)


def arr(limbs):
    return np.array(limbs, dtype=np.uint32)


def ptr(a):
    return a.ctypes.data_as(C.POINTER(C.c_uint32))


def val(limbs):
    return sum(int(x) << (29 * k) for k, x in enumerate(limbs))


def split(v):
    return [(v >> (29 * k)) & M29 for k in range(8)] + [v >> 232]


def check_reduced(out, t):
    """out is t / R mod p, below p + t / R, with limb 0 at most 2^29 and the others normalized."""
    assert int(out[0]) <= 1 << 29 and all(int(x) <= M29 for x in out[1:])
    assert (val(out) * R - t) % PF == 0 and val(out) <= PF + t // R


# limbs of a sum of two normalized values (one with limb 0 at 2^29), a normalized value, zero, one limb
BIG = [(1 << 30) - 1] + [(1 << 30) - 2] * 7 + [(1 << 23) - 1]
FULL = [1 << 29] + [M29] * 7 + [(1 << 22) - 1]


@pytest.mark.parametrize("a", [BIG, FULL, [0] * 9, [1] + [0] * 8, [0] * 8 + [(1 << 23) - 1], split(PF), split(8 * PF)])
@pytest.mark.parametrize("b", [BIG, FULL, [0] * 9, [1] + [0] * 8, split(PF), split(PF - 1)])
def test_products_at_the_limb_bounds(f9, a, b):
    out = arr([0] * 9)
    f9.f9_mul_limbs(ptr(arr(a)), ptr(arr(b)), ptr(out))
    check_reduced(out, val(a) * val(b))
    f9.f9_sqr_limbs(ptr(arr(a)), ptr(out))
    check_reduced(out, val(a) ** 2)


def test_products_random_limbs(f9):
    rng = random.Random(8)
    out = arr([0] * 9)
    for _ in range(500):
        a, b = ([rng.choice([0, M29, rng.randrange(1 << 29)]) for _ in range(8)] + [rng.randrange(1 << 22)]
                for _ in range(2))
        d = [2 * x for x in a]  # a normalized value by doubled limbs, as the partial round's last product
        f9.f9_mul_limbs(ptr(arr(b)), ptr(arr(d)), ptr(out))
        check_reduced(out, val(b) * val(d))


@pytest.mark.parametrize("u", ["top", "ones", "zero", "random"])
@pytest.mark.parametrize("v", ["top", "ones", "zero", "random"])
def test_partial_round_at_the_value_bounds(f9, u, v):
    rng = random.Random(9)
    top = (1 << 252) + (1 << 235)  # the bound a folded u keeps
    pick = {"top": lambda: top - 1, "ones": lambda: (1 << 252) - 1, "zero": lambda: 0,
            "random": lambda: rng.randrange(top)}
    for r in (1, 2, 57, 82):
        kd = arr([0] * 9)
        f9.f9_kd(r, ptr(kd))
        for x in (0, 1, PF, 7 * PF, rng.randrange(7 * PF)):
            uu, vv = pick[u](), pick[v]()
            U, V, X = arr(split(uu)), arr(split(vv)), arr(split(x))
            f9.f9_partial_round(ptr(U), ptr(V), ptr(X), r)
            y2 = 2 * pow(x * pow(R, -1, PF), 3, PF) * R  # 2 x^3 in Montgomery form
            assert val(V) == uu
            assert (val(U) - 4 * vv - 2 * uu - y2) % PF == 0 and val(U) < top
            assert (val(X) - uu - val(kd) + y2) % PF == 0 and val(X) < 7 * PF + (1 << 240)
            for out in (U, X):
                assert all(int(t) <= M29 for t in out[:8]) and int(out[8]) < 1 << 23
