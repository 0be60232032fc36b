"""Coherent emitters (phases zero) through the separable tiles, whose truncation is smooth in the emitter's
position and does not average out: the Laue closed form and near-field oracle rows, as for the other tiles."""
import numpy as np
import pytest

from conftest import K_UM
from gpu_util import rel_l2
from test_coherent_gpu import COHERENT_RTOL, LAUE_CASES, TOL_REV, _sc_sphere, box, forced, laue, lib  # noqa: F401

pytestmark = pytest.mark.gpu

TILES = range(17, 23)


@pytest.mark.parametrize("case", sorted(LAUE_CASES))
def test_laue_far_field(lib, case):  # noqa: F811
    import torch

    from oracle import Geometry

    (n0, pix, z), n, a = LAUE_CASES[case]
    expect = laue(Geometry(n0, n0, pix, z, K_UM), n, a)
    at = box(n, a)
    h = lib.Handle(n0, n0, pix, z, K_UM, precision=lib.PREC_FP32SPLIT)
    d = torch.from_numpy(at).cuda()
    checked = 0
    for tile in TILES:
        I, plan = forced(lib, h, d, tile)
        if plan["phase_bound"] <= TOL_REV:
            checked += 1
            assert rel_l2(I, expect) <= COHERENT_RTOL, (case, tile, plan)
    assert checked >= 1


@pytest.mark.parametrize("name", ["crystal", "coarse"])
def test_near_field_rows(lib, oracle_mod, name):  # noqa: F811
    """100000 simple-cubic sites in 10 nm, and 20000 in 30 nm where only tile 22 qualifies."""
    import torch

    from oracle import Geometry

    rng = np.random.default_rng(7200)
    if name == "crystal":
        g, sites, n = Geometry(512, 512, 75.0, 2e5, K_UM, nf=True), _sc_sphere(3e-4, 0.01), 100000
    else:
        g, sites, n = Geometry(256, 256, 100.0, 1e5, K_UM, nf=True), _sc_sphere(6e-4, 0.03), 20000
    at = np.c_[sites[rng.choice(len(sites), n, replace=False)], np.zeros(n)]
    rows = [0, g.n0 // 2 - 1, g.n0 // 2, 200]
    ref = np.abs(oracle_mod.field_c(g, at, rows=rows)) ** 2
    h = lib.Handle(g.n0, g.n1, g.pixelsize, g.detz, K_UM, nf=True, precision=lib.PREC_FP32SPLIT)
    d = torch.from_numpy(np.ascontiguousarray(at)).cuda()
    checked = 0
    for tile in [-1, *TILES]:
        I, plan = forced(lib, h, d, tile)
        if plan["phase_bound"] <= TOL_REV:
            assert tile >= 0 or plan["tile"] in TILES
            checked += 1
            assert rel_l2(I[rows], ref) <= COHERENT_RTOL, (tile, plan)
    assert checked >= 2
