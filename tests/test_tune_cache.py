"""The process-wide cache of tile shapes (alsvinn_amd/csrc/avh_tune.hpp), on the
CPU: a shape timed for one integrator's launches, or for a batch, is not handed
to another, and one timed on a solver that had stopped is not kept."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <set>
#include "avh_tune.hpp"
using namespace avh;
static int bad = 0;
#define CHECK(x) do { if (!(x)) { ++bad; printf("line %d: %s\n", __LINE__, #x); } } while (0)
static avh_config config(int eq, int recon, int flux, int integ) {
    avh_config c{};
    c.equation = eq;
    c.reconstruction = recon;
    c.flux = flux;
    c.integrator = integ;
    return c;
}
int main() {
    std::set<TuneKey> keys;
    int made = 0;
    for (int kind = 0; kind < 2; ++kind)
        for (int eq = 0; eq < 4; ++eq)
            for (int recon = 0; recon < 4; ++recon)
                for (int flux = 0; flux < 3; ++flux)
                    for (int integ = 0; integ < 3; ++integ)
                        for (long long n = 16; n < 18; ++n, ++made)
                            keys.insert(tune_key((TuneKind)kind, config(eq, recon, flux, integ), 2, {n, 33, 1}));
    CHECK((int)keys.size() == made);
    // an RK3 solver's choice is RK3's
    const avh_config rk3 = config(2, 1, 2, 2), rk2 = config(2, 1, 2, 1);
    tune_store(tune_key(TUNE_SOLVER, rk3, 2, {64, 64, 1}), 2, true);
    int s = -1;
    CHECK(tune_lookup(tune_key(TUNE_SOLVER, rk3, 2, {64, 64, 1}), &s) && s == 2);
    CHECK(!tune_lookup(tune_key(TUNE_SOLVER, rk2, 2, {64, 64, 1}), &s));
    CHECK(!tune_lookup(tune_key(TUNE_BATCH, rk3, 2, {64, 64, 1}), &s));
    // timed on the first stage alone: not kept
    tune_store(tune_key(TUNE_SOLVER, rk2, 2, {64, 64, 1}), 4, false);
    CHECK(!tune_lookup(tune_key(TUNE_SOLVER, rk2, 2, {64, 64, 1}), &s));
    tune_store(tune_key(TUNE_SOLVER, rk2, 2, {64, 64, 1}), 1, true);
    CHECK(tune_lookup(tune_key(TUNE_SOLVER, rk2, 2, {64, 64, 1}), &s) && s == 1);
    return bad ? 1 : 0;
}
"""


def test_choices_hold_for_what_was_timed(tmp_path):
    src = tmp_path / "tune.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "tune"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-I", os.path.join(ROOT, "alsvinn_amd", "csrc"), "-o",
                    str(exe), str(src)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
