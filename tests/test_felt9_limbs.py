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


def sval(limbs):
    return sum(int(x) << (29 * k) for k, x in enumerate(limbs.astype(np.int32)))


@pytest.mark.parametrize("x", ["plus", "minus", "mixed", "random"])
def test_signed_products_at_the_limb_bounds(f9, x):
    """A difference of two normalized values, limb 6 moved by up to 2^28 more, and its double."""
    rng = random.Random(10)
    top = [1 << 29] * 6 + [(1 << 29) + (1 << 28), 1 << 29, (1 << 21) - 1]
    for _ in range(1 if x in ("plus", "minus") else 200):
        limbs = [{"plus": 1, "minus": -1, "mixed": rng.choice([-1, 0, 1]), "random": rng.uniform(-1, 1)}[x] * t for t in top]
        a = np.array([int(t) for t in limbs], dtype=np.int32).view(np.uint32)
        d = np.array([2 * int(t) for t in limbs], dtype=np.int32).view(np.uint32)
        sq, out = arr([0] * 9), arr([0] * 9)
        f9.f9_sqr_signed(ptr(a), ptr(sq))
        check_reduced(sq, sval(a) ** 2)
        b = arr([1 << 29] + [M29] * 7 + [(1 << 20) - 1]) if x != "random" else sq
        f9.f9_mul_signed(ptr(b), ptr(d), ptr(out))
        t = sval(b) * sval(d)
        assert (sval(out) * R - t) % PF == 0 and t // R <= sval(out) <= PF + t // R + 1
        assert int(out[0]) <= 1 << 29 and all(int(v) <= M29 for v in out[1:8])


def test_partial_round_constants(f9):
    """The ranges that keep every 32-bit limb sum of the carry pass in place."""
    for r in range(1, 83):
        ku = arr([0] * 10)
        f9.f9_ku(r, ptr(ku))
        assert all(int(t) <= (1 << 29) - 8 for t in ku[:8]) and int(ku[8]) < 1 << 20
        assert int(ku[0]) >= 16 and int(ku[6]) >= 16 * (17 << 18)
        assert int(ku.astype(np.int32)[9]) in (0, 1 << 28, -(1 << 28))


@pytest.mark.parametrize("u", ["top", "ones", "zero", "random"])
@pytest.mark.parametrize("v", ["top", "ones", "zero", "random"])
def test_partial_round_at_the_value_bounds(f9, u, v):
    rng = random.Random(9)
    top = (1 << 252) + (1 << 235)  # the bound a folded u keeps
    pick = {"top": lambda: top - 1, "ones": lambda: (1 << 252) - 1, "zero": lambda: 0,
            "random": lambda: rng.randrange(top)}
    for r in range(1, 83):
        ku = arr([0] * 10)
        f9.f9_ku(r, ptr(ku))
        x6 = int(ku.astype(np.int32)[9]) << 174
        for x in (0, 1, PF, 3 * PF, -1, -PF, rng.randrange(3 * PF), -rng.randrange(PF)):
            uu, vv = pick[u](), pick[v]()
            limbs = split(abs(x))
            U, V = arr(split(uu)), arr(split(vv))
            X = np.array([t if x >= 0 else -t for t in limbs], dtype=np.int32).view(np.uint32)
            f9.f9_partial_round(ptr(U), ptr(V), ptr(X), r)
            y2 = 2 * pow(x * pow(R, -1, PF), 3, PF) * R  # 2 x^3 in Montgomery form
            assert val(V) == uu
            fold = (PF - (1 << 251))  # the share of p in ku's limbs 0 and 6
            assert (val(U) - 4 * vv - 2 * uu - y2 - val(ku[:9]) + fold) % PF == 0 and 0 < val(U) < top
            assert (sval(X) - uu + x6 + y2) % PF == 0 and -1.2 * PF < sval(X) < 3 * PF
            assert all(int(t) <= M29 for t in U[:8])
            assert all(abs(int(t)) <= (1 << 29) + ((1 << 28) if k == 6 else 0)
                       for k, t in enumerate(X.astype(np.int32)[:8]))
