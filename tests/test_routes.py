"""Every kernel of the stage's dispatch on the same grids, forward and
tangent-linear (CPU: the host build with the dispatch's limits moved, so that
small grids reach each kernel).

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

import numpy as np
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

# the tangent-linear run in FP64 and with FP32 pairs: values against the
# oracle's states, mixed tangents against the FP64 ones
CHILD_TL = """
import json, sys
import numpy as np
from oracle.pyoracle import Oracle
from smaug_amd.engine import Engine
from smaug_amd.params import npert
from tests.cases import compare, rel_l2, strat_case
ni, rkon, skew = json.loads(sys.argv[1])
rp, w, pos = strat_case(tuple(ni), ndim=len(ni), rkon=rkon)
rng = np.random.default_rng(3)
if skew:
    pos = pos * (1.0 + 1e-3 * rng.random(pos.shape))
k = npert(rp.ndim)
dw = rng.standard_normal((k, rp.ncells)) * np.sqrt((w[:k] ** 2).mean(axis=1))[:, None]
dbg = rng.standard_normal(w[k:].shape) * np.abs(w[k:])
orc = Oracle(rp, w, pos)
orc.step(2)
ref = orc.state()
out, tangents = {}, []
for prec in (0, 1):
    rp.precision = prec
    eng = Engine(rp, w, pos)
    eng.tl_begin(dw, dbg=dbg)
    eng.tl_step(2)
    v, d = eng.tl_get()
    out["mixed" if prec else "fp64"] = compare(rp, v, ref).tolist()
    tangents.append(d)
out["tangents"] = rel_l2(tangents[1], tangents[0]).tolist()
print(json.dumps(out))
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


def child(lib, align, case, code=CHILD):
    """The child's result (its last line) and the stage kernels it launched."""
    env = dict(os.environ, SMAUG_HIP_LIB=lib, EMU_ALIGN=align, EMU_TRACE="1", OMP_NUM_THREADS="2", PYTHONPATH=ROOT)
    p = subprocess.run([sys.executable, "-c", code, json.dumps(case)], cwd=ROOT, env=env, capture_output=True,
                       text=True, timeout=300)
    assert p.returncode == 0, f"{case}: {p.stdout[-500:]}\n{p.stderr[-2000:]}"
    ran = {k for k in ("tiled", "small", "wide", "general") if f"launch (k_rhs_{k}<" in p.stderr or f"launch k_rhs_{k}\n" in p.stderr}
    return json.loads(p.stdout.strip().splitlines()[-1]), ran


def worst(errs):
    """The largest of the errors (NaN if one of them is not finite: no bar holds)."""
    return float(np.max(np.where(np.isfinite(errs), errs, np.nan)))


def errors(lib, align, *case):
    return worst(child(lib, align, case)[0])


def test_worst_keeps_a_nan():
    assert worst([1e-16, 2e-16]) == 2e-16
    assert not worst([1e-16, float("nan")]) <= 1e-12 and not worst([float("inf"), 1e-16]) <= 1e-12


SIZES = [(12, 6, 6), (16, 8, 8), (17, 9, 12), (24, 7, 15), (32, 16, 8)]


@pytest.mark.parametrize("route", list(ROUTES))
@pytest.mark.parametrize("ni", SIZES)
def test_3d_grids(libs, route, ni):
    align = "start" if ni[0] % 2 else "end"
    errs, ran = child(libs[route], align, ("strat", ni, 1, 0, 0, 4, 0xFF))
    assert worst(errs) <= 1e-12 and ran == {route}
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
        errs, ran = child(libs["small"], "end", ("strat", (12, 6, 6), 0, 0, 0, 4, terms))
        assert worst(errs) <= 1e-12, hex(terms)
        assert ran == {kernel}, (hex(terms), ran)


@pytest.mark.parametrize("route,ni,skew", [("tiled", (17, 9, 12), 0), ("small", (17, 9, 12), 0), ("tiled", (17, 9, 12), 1),
                                           ("tiled", (24, 16, 18), 0), ("tiled", (17, 33), 0), ("tiled", (17, 33), 1)])
def test_tangent_kernels(libs, route, ni, skew):
    """The dual-number kernels: tiled and small, and k_rhs_general on
    positions that are no tensor product."""
    for align, rkon in (("end", 1), ("start", 0)):
        r, ran = child(libs[route], align, (ni, rkon, skew), CHILD_TL)
        # (FP64 pairs of a 3D grid take the tiled kernel on every route)
        assert ran == ({"general"} if skew else {"tiled", route}), ran
        assert worst(r["fp64"]) <= 1e-12, r
        assert worst(r["mixed"]) <= 1e-5, r
        assert worst(r["tangents"]) <= 1e-5, r


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
    for terms in (0x01, 0x02, 0x08, 0x10, 0x20, 0x40, 0x85, 0xFD):
        assert errors(libs["tiled"], "end", "strat", (17, 18), 1, 0, 0, 4, terms) <= 1e-12, hex(terms)
    for ni in ((12, 6), (16, 16), (17, 33), (31, 48)):
        assert errors(libs["tiled"], "end", "strat", ni, 1, 0, 0, 4, 0xFF) <= 1e-12, ni
        assert errors(libs["tiled"], "start", "strat", ni, 1, 0, 1, 4, 0xFF) <= 1e-12, ni
        assert errors(libs["tiled"], "end", "strat", ni, 0, 1, 0, 6, 0xFF) <= 1e-5, ni
    for n in (6, 16, 17):
        assert errors(libs["tiled"], "start", "ot", (n, n), 1, 0, 0, 0, 0xFF) <= 1e-12, n


@pytest.mark.gpu
@pytest.mark.parametrize("ni,rkon,mixed", [((4, 4, 4), 0, 0), ((5, 12, 4), 0, 0), ((12, 4, 5), 0, 1), ((40, 40, 40), 0, 0),
                                           ((41, 40, 40), 0, 0), ((40, 40, 40), 0, 1), ((64, 64, 33), 0, 1),
                                           ((187, 181, 190), 1, 0)])
def test_routes_on_the_gpu(ni, rkon, mixed):
    """The smallest grids, both sides of the limits in FP64 and FP32, and the
    wide kernel on odd sizes: rows that are not aligned, pairs of which one
    cell is interior, partial tiles along every axis, and the Runge-Kutta
    combination of pairs."""
    from oracle.pyoracle import Oracle
    from smaug_amd.engine import Engine
    from tests.cases import compare, strat_case

    rp, w, pos = strat_case(ni, rkon=rkon)
    print("routes:", ni, "rk" if rkon else "single stage", "mixed" if mixed else "fp64", flush=True)
    orc = Oracle(rp, w, pos)
    orc.step(1)
    ref = orc.state()
    orc.close()
    rp.precision = mixed
    eng = Engine(rp, w, pos)
    eng.step(1)
    got = eng.state()
    eng.close()
    assert worst(compare(rp, got, ref)) <= (1e-5 if mixed else 1e-12)
