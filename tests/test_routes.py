"""Every kernel of the stage's dispatch on the same grids (CPU: the host build
with the dispatch's limits moved, so that small grids reach each kernel).

launch_tiled_t sends a tensor-product grid to k_rhs_small (all boxes of a tile
in LDS), k_rhs_tiled or k_rhs_wide (FP64, two cells per thread) by its number
of tiles, and any other grid to k_rhs_general.  Each is compared with the
oracle on grids around the tiles' edges: less than one, whole tiles, one
cell more and less, odd sizes, a single tile along an axis.  The bars are the
suite's own: relative L2 per variable of 1e-12 in FP64 (sums in another order)
and 1e-5 with FP32 stencils."""
from __future__ import annotations

import json
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HERE = os.path.join(ROOT, "tests", "hostemu")
ROUTES = {"tiled": (0, 1 << 30), "small": (1 << 20, 1 << 30), "wide": (0, 1)}

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")

CHILD = """
import json, sys
import numpy as np
from oracle.pyoracle import Oracle
from smaug_amd.engine import Engine
from tests.cases import compare, ot_case, strat_case
kind, ni, rkon, mixed, skew, bc, terms = json.loads(sys.argv[1])
if kind == "ot":
    rp, w, pos = ot_case(ni[0], rkon)
else:
    rp, w, pos = strat_case(tuple(ni), ndim=len(ni), rkon=rkon)
    rp.bcu = [bc] * 3
    rp.bcl = [bc] * 3
rp.terms = terms
if skew:  # positions that are no tensor product
    pos = pos * (1.0 + 1e-3 * np.random.default_rng(3).random(pos.shape))
orc = Oracle(rp, w, pos)
orc.step(2)
ref = orc.state()
rp.precision = int(mixed)
eng = Engine(rp, w, pos)
eng.step(2)
print(json.dumps(compare(rp, eng.state(), ref).tolist()))
"""


@pytest.fixture(scope="module")
def libs(tmp_path_factory):
    csrc = os.path.join(ROOT, "smaug_amd", "csrc")
    src = [os.path.join(HERE, "emu.cpp")] + [
        os.path.join(csrc, f) for f in ("smaug_kernels.hip", "smaug_rhs.hip", "smaug_adj.hip", "smaug_host.hip", "smaug_io.cpp")]
    out, jobs = {}, []
    for name, (cus, wide) in ROUTES.items():
        out[name] = str(tmp_path_factory.mktemp("routes") / f"{name}.so")
        jobs.append(subprocess.Popen(
            ["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-w", f"-DSMAUG_CUS={cus}", f"-DSMAUG_WIDE_TILES={wide}",
             "-I", HERE, "-o", out[name], "-x", "c++", *src]))
    assert all(p.wait() == 0 for p in jobs)
    return out


def child(lib, align, case, **env):
    env = dict(os.environ, SMAUG_HIP_LIB=lib, EMU_ALIGN=align, OMP_NUM_THREADS="2", PYTHONPATH=ROOT, **env)
    p = subprocess.run([sys.executable, "-c", CHILD, json.dumps(case)], cwd=ROOT, env=env, capture_output=True,
                       text=True, timeout=300)
    assert p.returncode == 0, f"{case}: {p.stdout[-500:]}\n{p.stderr[-2000:]}"
    return p


def errors(lib, align, *case):
    return max(json.loads(child(lib, align, case).stdout.strip().splitlines()[-1]))


SIZES = [(12, 6, 6), (16, 8, 8), (17, 9, 12), (24, 7, 15), (32, 16, 8)]


@pytest.mark.parametrize("route", list(ROUTES))
@pytest.mark.parametrize("ni", SIZES)
def test_3d_grids(libs, route, ni):
    align = "start" if ni[0] % 2 else "end"
    assert errors(libs[route], align, "strat", ni, 1, 0, 0, 4, 0xFF) <= 1e-12
    assert errors(libs[route], align, "strat", ni, 0, 1, 0, 4, 0xFF) <= 1e-5


@pytest.mark.parametrize("route", list(ROUTES))
def test_3d_boundaries_terms_and_other_grids(libs, route):
    for bc in (3, 5, 7):  # cont, fixed, asymm
        assert errors(libs[route], "end", "strat", (17, 12, 10), 0, 0, 0, bc, 0xFF) <= 1e-12, bc
    for terms in (0x01, 0x08, 0x10, 0x22, 0x20, 0x02, 0x40, 0x84):
        assert errors(libs[route], "end", "strat", (17, 12, 10), 0, 0, 0, 4, terms) <= 1e-12, hex(terms)
    assert errors(libs[route], "end", "strat", (17, 12, 10), 1, 0, 1, 4, 0xFF) <= 1e-12
    assert errors(libs[route], "start", "strat", (17, 12, 10), 1, 1, 1, 4, 0xFF) <= 1e-5


def test_small_grids_by_terms(libs):
    """k_rhs_small stages every box of a tile; where the term mask leaves out
    the phases of v_f and b_f, the tiled kernel runs, which stages less."""
    flux, eterm, grav, hrho, he, hmom, hb, src = (1 << k for k in range(8))
    for terms, kernel in ((0, "tiled"), (flux | grav | src, "tiled"), (flux | hrho | he, "tiled"), (flux | eterm, "small"),
                          (hmom, "small"), (hb, "small"), (0xFF, "small")):
        p = child(libs["small"], "end", ("strat", (12, 6, 6), 0, 0, 0, 4, terms), EMU_TRACE="1")
        assert max(json.loads(p.stdout.strip().splitlines()[-1])) <= 1e-12, hex(terms)
        ran = {k for k in ("tiled", "small", "wide", "general") if f"launch (k_rhs_{k}" in p.stderr}
        assert ran == {kernel}, (hex(terms), ran)


# 4 and 5 interior cells along an axis (the smallest the engine takes): a cell
# there feeds a ghost on either side, two in all.  (The stratified atmosphere
# on so few cells along dim 0 is stable with the single-stage scheme only: RK4
# takes the oracle to negative densities within two steps.)
SMALLEST = [(4, 4, 4), (5, 5, 5), (12, 4, 5), (5, 12, 4), (4, 5, 12)]


@pytest.mark.parametrize("route", list(ROUTES))
def test_smallest_3d_grids(libs, route):
    for ni in SMALLEST:
        for bc in (3, 4, 5, 6, 7):  # cont, contcd4, fixed, symm, asymm
            assert errors(libs[route], "end", "strat", ni, 0, 0, 0, bc, 0xFF) <= 1e-12, (ni, bc)
        assert errors(libs[route], "start", "strat", ni, 0, 1, 0, 4, 0xFF) <= 1e-5, ni
    assert errors(libs[route], "start", "strat", (12, 4, 5), 1, 0, 0, 4, 0xFF) <= 1e-12


def test_smallest_2d_grids(libs):
    for ni in ((4, 4), (5, 4), (4, 17), (16, 5)):
        for bc in (3, 4, 5, 6, 7):
            assert errors(libs["tiled"], "end", "strat", ni, int(ni[0] > 8), 0, 0, bc, 0xFF) <= 1e-12, (ni, bc)
    for n in (4, 5):
        assert errors(libs["tiled"], "end", "ot", (n, n), 1, 0, 0, 0, 0xFF) <= 1e-12, n


def test_2d_grids(libs):
    for ni in ((12, 6), (16, 16), (17, 33), (31, 48)):
        assert errors(libs["tiled"], "end", "strat", ni, 1, 0, 0, 4, 0xFF) <= 1e-12, ni
        assert errors(libs["tiled"], "start", "strat", ni, 1, 0, 1, 4, 0xFF) <= 1e-12, ni
        assert errors(libs["tiled"], "end", "strat", ni, 0, 1, 0, 6, 0xFF) <= 1e-5, ni
    for n in (6, 16, 17):
        assert errors(libs["tiled"], "start", "ot", (n, n), 1, 0, 0, 0, 0xFF) <= 1e-12, n


@pytest.mark.gpu
@pytest.mark.parametrize("ni,mixed", [((4, 4, 4), 0), ((5, 12, 4), 0), ((12, 4, 5), 1), ((40, 40, 40), 0), ((41, 40, 40), 0), ((40, 40, 40), 1), ((64, 64, 33), 1),
                                      ((184, 184, 184), 0)])
def test_routes_on_the_gpu(ni, mixed):
    """The smallest grids, both sides of the limits in FP64 and FP32, and the
    wide kernel on a grid whose rows are not aligned."""
    from oracle.pyoracle import Oracle
    from smaug_amd.engine import Engine
    from tests.cases import compare, strat_case

    rp, w, pos = strat_case(ni, rkon=0)
    print("routes:", ni, "mixed" if mixed else "fp64", flush=True)
    orc = Oracle(rp, w, pos)
    orc.step(1)
    ref = orc.state()
    orc.close()
    rp.precision = mixed
    eng = Engine(rp, w, pos)
    eng.step(1)
    got = eng.state()
    eng.close()
    assert compare(rp, got, ref).max() <= (1e-5 if mixed else 1e-12)
