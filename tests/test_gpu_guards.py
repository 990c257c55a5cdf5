"""The shared-reciprocal path of the stage kernels rests on range checks per
launch, per cell and per interface; whatever a check lets through or turns
away must give the oracle's bits.  States are drawn with magnitudes on both
sides of each bound (momenta about 2^-600 and 2^-390 and at 0, densities about
2^-90, pressures about 2^-300, sums of magnitudes about 2^85), with cells of
ordinary size between them, so that one tile holds both kinds."""
import ctypes

import numpy as np
import pytest

import alsvinn_amd
from alsvinn_amd import _abi
from alsvinn_amd.simulator import default_context
from tests.cases import smooth_state
from tests.test_gpu_parity import make_pair

pytestmark = pytest.mark.gpu

KINDS = {5: "star quotients, denominators +-[2^-150, 2^150]", 6: "1/d, d in [2^-53, 2^348]"}


@pytest.mark.parametrize("kind", sorted(KINDS))
def test_star_and_reciprocal_shortcuts_bitwise(kind):
    bad = ctypes.c_int64(-1)
    first = (ctypes.c_double * 2)()
    print("case arith kind", kind, KINDS[kind], flush=True)
    _abi.check(alsvinn_amd.load().avh_arith_selftest(default_context()._h, kind, 0xBEEF + kind, 100_000_000,
                                                     ctypes.byref(bad), first))
    assert bad.value == 0, "%d mismatches, e.g. operands %r %r" % (bad.value, first[0], first[1])


BOUNDS = {
    "tiny momenta": lambda r, q: _momenta(r, q, (-640, -560)),
    "small momenta": lambda r, q: _momenta(r, q, (-400, -380)),
    "signed zero momenta": lambda r, q: _zeros(r, q),
    "small densities": lambda r, q: _scale(r, q, (-96, -84)),
    "small pressures": lambda r, q: _pressure(r, q, (-310, -290)),
    "large cells": lambda r, q: _scale(r, q, (80, 90)),
    "mixed": lambda r, q: _mixed(r, q),
}


def _pick(r, q, share=0.15):
    return r.random(q.shape[1:]) < share


def _pow2(r, shape, e):
    return np.ldexp(0.5 + 0.5 * r.random(shape), r.integers(e[0], e[1], size=shape))


def _momenta(r, q, e):
    for v in range(1, q.shape[0] - 1):
        at = _pick(r, q)
        q[v][at] = (_pow2(r, q[v].shape, e) * r.choice([-1.0, 1.0], size=q[v].shape))[at]


def _zeros(r, q):
    for v in range(1, q.shape[0] - 1):
        at = _pick(r, q, 0.5)
        q[v][at] = r.choice([-0.0, 0.0], size=q[v].shape)[at]


def _scale(r, q, e):
    at = _pick(r, q)
    q[:, at] = (q * _pow2(r, q.shape[1:], e)[None])[:, at]


def _pressure(r, q, e):
    # cells at rest, so that the energy is the pressure's
    at = _pick(r, q)
    for v in range(1, q.shape[0] - 1):
        q[v][at] = 0.0
    q[-1][at] = _pow2(r, q.shape[1:], e)[at]


def _mixed(r, q):
    for f in (_zeros, lambda a, b: _momenta(a, b, (-1070, -350)), lambda a, b: _scale(a, b, (-100, 95))):
        f(r, q)


GRIDS = [("euler1", (97,)), ("euler2", (45, 34)), ("euler3", (19, 17, 9))]


@pytest.mark.parametrize("bound", sorted(BOUNDS))
@pytest.mark.parametrize("equation,n", GRIDS)
def test_guard_bounds_bitwise(equation, n, bound):
    from oracle import pyoracle
    r = np.random.default_rng(len(bound) * 100 + len(n))
    for recon in ("weno2", "eno3", "none"):
        for flux in ("hll3", "hll"):
            q = np.ascontiguousarray(smooth_state(equation, n, seed=len(bound) + len(recon), jump=True))
            with np.errstate(all="ignore"):
                BOUNDS[bound](r, q)
            print("case guard", bound, equation, n, recon, flux, flush=True)
            o, h = make_pair(pyoracle, equation, recon, flux, "forwardeuler", "periodic", n, 0.4)
            o.set_interior(q)
            U = o.get_state()
            out_o, ws_o = pyoracle.compute_flux(o.cfg, U, np.zeros_like(U))
            want = np.ascontiguousarray(o.interior(out_o)).view(np.uint64)
            for shape in range(7 if len(n) == 3 else (5 if len(n) == 2 else 2)):
                h.set_tile_shape(shape)
                h.set_interior(q)
                out_h, ws_h = h.compute_flux()
                got = np.ascontiguousarray(out_h).view(np.uint64)
                nan = np.isnan(np.ascontiguousarray(o.interior(out_o)))
                assert np.array_equal(np.isnan(out_h), nan)
                assert np.array_equal(np.asarray(ws_h).view(np.uint64), np.asarray(ws_o).view(np.uint64))
                assert np.array_equal(got[~nan], want[~nan]), "shape %d" % shape


BURGERS = {"zeros": None, "tiny": (-1070, -590), "about 2^-600": (-606, -594), "about 2^85": (80, 90),
           "all": (-1070, 200)}


@pytest.mark.parametrize("bound", sorted(BURGERS))
@pytest.mark.parametrize("n", [(97,), (45, 34), (19, 17, 9)])
def test_burgers_guard_bounds_bitwise(n, bound):
    """Burgers' WENO2 weights on both sides of the cell check: the net flux on
    every tile shape, and in 1D a step (the one-workgroup path)."""
    from oracle import pyoracle
    r = np.random.default_rng(len(bound) * 10 + len(n))
    q = np.ascontiguousarray(smooth_state("burgers", n, seed=len(bound), jump=True))
    at = _pick(r, q)
    q[0][at] = (r.choice([-0.0, 0.0], size=q[0].shape) if BURGERS[bound] is None else
                _pow2(r, q[0].shape, BURGERS[bound]) * r.choice([-1.0, 1.0], size=q[0].shape))[at]
    print("case burgers guard", bound, n, flush=True)
    o, h = make_pair(pyoracle, "burgers", "weno2", "godunov", "rungekutta3", "periodic", n, 0.4)
    o.set_interior(q)
    U = o.get_state()
    out_o, ws_o = pyoracle.compute_flux(o.cfg, U, np.zeros_like(U))
    want = np.ascontiguousarray(o.interior(out_o)).view(np.uint64)
    for shape in range((2, 5, 7)[len(n) - 1]):
        h.set_tile_shape(shape)
        h.set_interior(q)
        out_h, ws_h = h.compute_flux()
        assert np.array_equal(np.asarray(ws_h).view(np.uint64), np.asarray(ws_o).view(np.uint64))
        assert np.array_equal(np.ascontiguousarray(out_h).view(np.uint64), want), "shape %d" % shape
    h.set_tile_shape(-1)
    h.set_interior(q)
    h.perform_step()
    o.step()
    assert np.array_equal(h.get_interior().view(np.uint64),
                          np.ascontiguousarray(o.interior(o.get_state())).view(np.uint64))
