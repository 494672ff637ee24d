"""The kernels' FP64 quotient and square root (phlx_fp64.hpp), built for the
host with hardware seeds of random error up to their bound of 2^-24, against
IEEE division and sqrt: the same bits over the exponents that flows have and
for every zero, infinity and NaN; a neighbour at most where the exact result
lies within 2^-45 ulp of the midpoint of two numbers, and where the remainder
underflows.
"""
import ctypes
import itertools
import math
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def ops(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fp64") / "ops.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-fPIC", "-shared", "-o", so,
                    os.path.join(HERE, "fp64_ops_host.cpp")], check=True)
    lib = ctypes.CDLL(so)
    d, n = ctypes.c_double, ctypes.c_long
    lib.set_seed_error.argtypes, lib.set_seed_error.restype = [d], None
    lib.quotient.argtypes, lib.quotient.restype = [d, d], d
    lib.reciprocal.argtypes, lib.reciprocal.restype = [d], d
    lib.root.argtypes, lib.root.restype = [d], d
    for f in (lib.random_mismatches, lib.smallest_operands):
        f.argtypes, f.restype = [n], n
    lib.hardest_quotients.argtypes = [n, ctypes.POINTER(n)]
    lib.hardest_quotients.restype = n
    lib.hardest_roots.argtypes, lib.hardest_roots.restype = [ctypes.POINTER(n)], n
    return lib


def _same(a, b):
    return (math.isnan(a) and math.isnan(b)) or (a == b and
                                                 math.copysign(1, a) == math.copysign(1, b))


def _ieee(a, b):
    if b != 0.0:
        return a / b
    if a == 0.0 or math.isnan(a) or math.isnan(b):
        return math.nan
    return math.copysign(math.inf, a) * math.copysign(1.0, b)


SPECIAL = [0.0, 1.0, 3.0, 1e-280, 1e280, math.inf]


@pytest.mark.parametrize("eps", [0.0, 2.0 ** -24, -(2.0 ** -24)])
def test_special_values(ops, eps):
    ops.set_seed_error(eps)
    values = SPECIAL + [-v for v in SPECIAL] + [math.nan]
    for a, b in itertools.product(values, values):
        if 1e-285 < abs(_ieee(a, b)) < 1e285 or not math.isfinite(a * b) or a * b == 0.0:
            assert _same(ops.quotient(a, b), _ieee(a, b)), (a, b)
    for b in values:
        assert _same(ops.reciprocal(b), _ieee(1.0, b)), b
    for x in values:
        want = math.nan if x < 0.0 or math.isnan(x) else math.sqrt(x)
        assert _same(ops.root(x), want), x
    assert _same(ops.root(-0.0), -0.0)


def test_random_operands_bitwise(ops):
    assert ops.random_mismatches(2_000_000) == 0


def test_hardest_roundings(ops):
    n = ctypes.c_long()
    assert ops.hardest_quotients(200_000, ctypes.byref(n)) <= 1 and n.value > 100_000
    assert ops.hardest_roots(ctypes.byref(n)) <= 1 and n.value > 1000


def test_underflowing_remainders(ops):
    assert ops.smallest_operands(500_000) <= 1
