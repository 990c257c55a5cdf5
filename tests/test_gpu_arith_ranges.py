"""The self-test's kind 5 over the ranges of the flux functions' quotients, to
their ends: HLL's denominators to 2^180, HLL3's transverse numerators down to
2^-919 with quotients down to 2^-999 (the range of the draws is in
include/alsvinn_hip.h), with other seeds than test_gpu_guards.py; and the header
describes every kind there is."""
import ctypes
import os
import re

import pytest

import alsvinn_amd
from alsvinn_amd import _abi
from alsvinn_amd.simulator import default_context

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = open(os.path.join(ROOT, "alsvinn_amd", "csrc", "avh_capi.hip")).read()
GUARDS = open(os.path.join(ROOT, "alsvinn_amd", "csrc", "avh_physics.hpp")).read()


def test_draws_reach_the_guards():
    """Each guard's bound, as the flux functions state it, is an end of a draw."""
    draws = SOURCE[SOURCE.index("kind == ARITH_DIV_FLUX"):SOURCE.index("kind == ARITH_DIV_ONE")]
    ends = {tuple(map(int, m)) for m in re.findall(r"draw_double\(r[01], (-?\d+), (-?\d+)\)", draws)}
    assert {(-100, 180), (-701, 456), (-150, 80), (-919, 268), (-100, 150), (-800, 630)} <= ends
    text = " ".join(GUARDS.split())
    for bound in ("den in [2^-100, 2^180]", "[2^-701, 2^456]", "-aa in [2^-150, 2^80]", "[2^-919, 2^268]",
                  "|s_m - s_k| in [2^-100, 2^150]"):
        assert bound in text.replace("// ", ""), bound
    header = open(os.path.join(ROOT, "include", "alsvinn_hip.h")).read()
    doc = header[:header.index("avh_status avh_arith_selftest")].rsplit("/*", 1)[1]
    for kind in range(7):
        assert "%d: " % kind in doc


@pytest.mark.gpu
@pytest.mark.parametrize("seed", [11, 12])
def test_flux_quotients_bitwise(seed):
    bad = ctypes.c_int64(-1)
    first = (ctypes.c_double * 2)()
    print("case flux quotients", seed, flush=True)
    _abi.check(alsvinn_amd.load().avh_arith_selftest(default_context()._h, 5, seed, 200_000_000, ctypes.byref(bad),
                                                     first))
    assert bad.value == 0, "%d mismatches, e.g. operands %r %r" % (bad.value, first[0], first[1])
