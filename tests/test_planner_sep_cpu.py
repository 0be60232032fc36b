"""The planner's tables of the separable tiles against an evaluation of every pixel in FP64 (no GPU).

planner_sep_tables looks at the corners of every rectangle (and its edges' ends) and adds 5%; the kernels use
all of its pixels.  tests/host_asan/planner_sep_check.cpp, built with the sanitizers, evaluates the mixed
remainder, its parts and the column phases at every pixel.
"""
import json
import os
import shutil
import subprocess

import numpy as np
import pytest

from conftest import K_UM
from test_planner_cpu import CASES

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "tests", "host_asan", "planner_sep_check.cpp")
TOL = 5e-6
DETECTORS = [args for args, _ in CASES] + [
    dict(n0=256, n1=256, pixelsize=100.0, detz=1e5),                                          # 16 x 16, second order
    dict(n0=333, n1=211, pixelsize=55.0, detz=1.5e5, detoffset=(900.0, -650.0), detangles=(0.03, 0.1)),
    dict(n0=70, n1=135, pixelsize=75.0, detz=2e5, detoffset=(9000.0, -15000.0), detangles=(0.3, -0.5)),
    dict(n0=1, n1=2049, pixelsize=75.0, detz=2e5),
    dict(n0=1, n1=1, pixelsize=75.0, detz=2e5),
    dict(n0=64, n1=48, pixelsize=300.0, detz=1e5),
    dict(n0=64, n1=64, pixelsize=2000.0, detz=1e4),                                           # past the series
]
EXTENTS = [0.002, 0.01, 0.03, 0.1]


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    if shutil.which("g++") is None or not os.path.exists("/opt/rocm/include/hip/hip_runtime.h"):
        pytest.skip("needs g++ and the ROCm headers")
    exe = str(tmp_path_factory.mktemp("planner_sep") / "planner_sep_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fno-omit-frame-pointer", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=all", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-ffp-contract=off",
                    "-Wall", "-Wextra", "-Wno-unknown-pragmas", SRC, "-o", exe], check=True)
    return exe


def _plan(driver, args, nf, secondorder=False, summode=0):
    from oracle import Geometry

    g = Geometry(args["n0"], args["n1"], args["pixelsize"], args["detz"], K_UM, nf=nf, secondorder=secondorder,
                 detoffset=args.get("detoffset", (0.0, 0.0)), detangles=args.get("detangles", (0.0, 0.0)))
    M = np.asarray(g.M, dtype=np.float64).ravel()
    line = " ".join(str(v) for v in (
        g.n0, g.n1, repr(float(g.pixelsize)), repr(float(g.detz)), repr(float(g.k)), repr(float(g.detoffset[0])),
        repr(float(g.detoffset[1])), int(nf), 0, int(secondorder), int(g.rot), *(repr(float(v)) for v in M), TOL, summode,
        len(EXTENTS), *(repr(v) for v in EXTENTS)))
    out = subprocess.run([driver], input=line + "\n", capture_output=True, text=True,
                         env=dict(os.environ, ASAN_OPTIONS="halt_on_error=1:abort_on_error=1", UBSAN_OPTIONS="halt_on_error=1"))
    assert out.returncode == 0, out.stderr[-3000:]
    return json.loads(out.stdout)


@pytest.mark.parametrize("args", DETECTORS, ids=lambda a: "%dx%d_%g_%g%s" % (
    a["n0"], a["n1"], a["pixelsize"], a["detz"], "_rot" if a.get("detangles") else ""))
def test_tables_bound_every_pixel(driver, args):
    r = _plan(driver, args, True)
    noise = 2.0**-50 * r["krev"]  # of FP64 differences of unit vectors
    for t, b in zip(r["tables"], r["brute"]):
        if t["mixed"] is None:  # past the series: no tile of this rectangle is taken, its entries are not read
            assert t["rest"] is None and t["off"] is None and t["fourth"] is None
            continue
        for key in ("line", "mixed", "rest", "off", "fourth", "du", "dR"):
            slack = 2.0**-50 * (args["detz"] if key == "dR" else 1.0) if key in ("du", "dR") else noise
            assert b[key] <= t[key] + slack, (key, t[key], b[key])
        # the kernel's FP32 series: its rounding (2^-20 of the largest remainder) and its fifth order
        # (e < 0.01: 1e-2^4 of it); FP64's own noise
        assert b["series"] <= 2e-6 * b["mixed"] + noise, (b["series"], b["mixed"])
        # not vacuous: the corners are where the remainder is largest
        assert t["mixed"] <= 1.0501 * b["mixed"] + noise


@pytest.mark.parametrize("nf,secondorder,summode", [(True, False, 0), (False, False, 0), (False, True, 0), (True, False, 1)])
def test_rule_follows_the_bounds(driver, nf, secondorder, summode):
    some = 0
    for args in DETECTORS:
        r = _plan(driver, args, nf, secondorder, summode)
        for rho, e in zip(EXTENTS, r["extents"]):
            for v in range(17, 23):
                t = r["brute"][{17: 0, 18: 0, 19: 1, 20: 1, 21: 2, 22: 2}[v]]
                ok = e["bound%d" % v] is not None and e["bound%d" % v] <= TOL
                assert (v in e["eligible"]) == (ok and not summode), (args, rho, v)
                if not ok:
                    continue
                some += 1
                # what the tile drops at its worst pixel, of a phasor exp(i M)
                M = 2 * np.pi * rho * t["mixed"]
                if v == 22:
                    drop = M**3 / 6 + M * 2 * np.pi * rho * t["rest"]
                else:
                    drop = M**2 / 2 + (0 if v in (18, 20) else 2 * np.pi * rho * t["off"])
                assert drop / (2 * np.pi) <= e["trunc%d" % v] * (1 + 1e-6) + 1e-15
                assert e["trunc%d" % v] <= 1.4e-6 and e["trunc%d" % v] <= e["bound%d" % v]
            sides = [s for s in (32, 16) if e["adjoint%d" % s] is not None and e["adjoint%d" % s] <= TOL]
            assert e["side"] == (sides[0] if sides else 0)
        # 4 has no kernel, 16 is no variant, 23 is past the last
        want = [0] * 24
        want[4], want[16], want[23] = -5, -1, -1
        assert r["option"] == want
    assert some > 20 or summode
