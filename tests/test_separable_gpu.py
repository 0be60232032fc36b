"""The separable forward tiles (matrix products over the emitters) against the FP64 oracle."""
import numpy as np
import pytest

from conftest import K_UM
from gpu_util import atoms_ball, fp64_tol, make_handle, rel_l2, run

pytestmark = pytest.mark.gpu

TILES = range(17, 23)  # 32 x 32, 32 x 64 and 16 x 16 pixels per wave, remainder along two directions or in full


@pytest.fixture(scope="module")
def lib():
    import torch

    from idi_amd import _lib

    assert torch.cuda.is_available()
    _lib.load()
    return _lib


def _check(f, ref, g, plan, amp_sum, what):
    """Per pixel: the planner's phase bound for every term, the FP32 roundings of the sums (at most 192
    matrix instructions add into one between two merges) and the oracle's own rounding of k |r_p|.
    A variant that the planner would not pick (it reports no bound) is not checked."""
    if not np.isfinite(plan["phase_bound"]):
        return
    assert plan["phase_bound"] <= 5e-6, (what, plan)
    tol = (2 * np.pi * plan["phase_bound"] + 192 * 2.0**-24 + fp64_tol(g)) * amp_sum
    err = np.abs(f - ref).max()
    assert err <= tol, (what, err, tol)


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("shape", [(1, 1), (31, 33), (64, 128), (65, 129)])
def test_edges_of_tiles_and_steps(lib, oracle_mod, tile, shape):
    """Detectors at and one past the edges of the wave and workgroup tiles; emitter counts at and around a
    step, a staging round and a merge of the sums; splits; amplitudes over nine decades.  At 0.5 m every
    variant meets the bound, at 0.2 m variant 19 (two directions over 32 x 64 pixels) may not."""
    from oracle import Geometry

    rng = np.random.default_rng(50)
    for z in (2e5, 5e5):
        g = Geometry(*shape, 75.0, z, K_UM, nf=True, detoffset=(1500.0, -2200.0))
        for n in (1, 7, 16, 33, 255, 257, 513, 1030):
            at = atoms_ball(rng, n, 0.01)
            amp = 10.0 ** rng.uniform(-6, 3, n) if n % 2 else None
            ref = oracle_mod.field_c(g, at, amp)
            for split in ((1, 3) if n > 300 else (1,)):
                f, h = run(lib, g, at, amp, tile=tile, split=split)
                p = h.plan()
                assert (p["tile"], p["split"], p["fallback"]) == (tile, split, 0)
                assert z == 2e5 or np.isfinite(p["phase_bound"])
                _check(f, ref, g, p, n if amp is None else amp.sum(), (tile, shape, n, split))


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("mode", ["nf", "nf scale amp", "ff", "ff secondorder", "ff scale amp", "nf rot"])
def test_phase_models(lib, oracle_mod, tile, mode):
    from oracle import Geometry

    rng = np.random.default_rng(51)
    rot = "rot" in mode
    g = Geometry(70, 135, 75.0, 2e5, K_UM, detoffset=(900.0, -1500.0) if rot else (0.0, 0.0),
                 detangles=(0.05, -0.08) if rot else (0.0, 0.0), nf=mode.startswith("nf"), scale="scale" in mode,
                 secondorder="secondorder" in mode)
    at = atoms_ball(rng, 700, 0.01)
    amp = rng.uniform(0.5, 1.0, 700) if "amp" in mode else None
    ref = oracle_mod.field_c(g, at, amp)
    f, h = run(lib, g, at, amp, tile=tile, split=2)
    total = 700 if amp is None else amp.sum()
    _check(f, ref, g, h.plan(), total / (2e5 if g.scale else 1.0), (tile, mode))
    I, _ = run(lib, g, at, amp, kind=lib.OUT_INTENSITY, tile=tile, split=1)
    assert rel_l2(I, np.abs(ref) ** 2) <= 1e-4


@pytest.mark.parametrize("tile", TILES)
def test_batched_equals_single_shot(lib, oracle_mod, tile):
    """The persistent kernel against the single-shot one of the same tile without a split, bit for bit:
    uneven shots, one empty, a detector that ends inside a tile."""
    import torch

    from oracle import Geometry

    rng = np.random.default_rng(53)
    g = Geometry(70, 135, 50.0, 5e5, K_UM, nf=True)
    sizes = [700, 0, 1, 1500, 513]
    shots = [atoms_ball(rng, n, 0.01) for n in sizes]
    amps = [rng.uniform(0.5, 1.0, n) for n in sizes]
    offsets = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    hb, hs = make_handle(lib, g, 1), make_handle(lib, g, 1)
    for h in (hb, hs):
        h.set_option(lib.OPT_TILE, tile)
        h.set_option(lib.OPT_SPLIT, 1)
    cat, acat = torch.from_numpy(np.concatenate(shots)).cuda(), torch.from_numpy(np.concatenate(amps)).cuda()
    for amp in (None, acat):
        out = hb.forward_batched(cat, offsets, amp, extent=0.01).cpu().numpy()
        assert hb.plan()["tile"] == tile and hb.plan()["phase_bound"] <= 5e-6
        for s, at in enumerate(shots):
            if sizes[s] == 0:
                assert np.count_nonzero(out[s]) == 0
                continue
            a = None if amp is None else torch.from_numpy(amps[s]).cuda()
            single = hs.forward(torch.from_numpy(at).cuda(), a, extent=0.01).cpu().numpy()
            np.testing.assert_array_equal(out[s], single)


def test_rule(lib, oracle_mod):
    """From 5e8 pairs on a field (an intensity from 1e8) takes a separable tile where one meets the bound,
    below it stays on the others; the loss-and-gradient call never does; a geometry whose remainder is too large keeps the
    other tiles; an emitter at the origin (no extent) is fine."""
    import torch

    from oracle import Geometry

    rng = np.random.default_rng(52)
    g = Geometry(256, 256, 75.0, 2e5, K_UM, nf=True)
    h = make_handle(lib, g, lib.PREC_FP32SPLIT)
    for n, sep in ((8192, True), (8191, False)):
        at = atoms_ball(rng, n, 0.01)
        d = torch.from_numpy(at).cuda()
        h.forward(d, None, None, lib.OUT_INTENSITY, 0.01)
        assert h.plan()["tile"] >= 17
        f = h.forward(d, None, None, lib.OUT_FIELD, 0.01).cpu().numpy()
        assert (h.plan()["tile"] >= 17) == sep, (n, h.plan())
        rows = [0, 101, 255]
        assert rel_l2(f[rows], oracle_mod.field_c(g, at, rows=rows)) <= 1e-4
    T = torch.rand((256, 256), dtype=torch.float32, device="cuda")
    at = atoms_ball(rng, 8192, 0.01)
    d = torch.from_numpy(at).cuda()
    field = torch.empty((256, 256), dtype=torch.complex64, device="cuda")
    h.loss_grad_l2(d, T, None, 0.01, field=field)
    f2 = h.forward(d, None, None, lib.OUT_FIELD, 0.01)
    assert h.plan()["tile"] >= 17
    assert rel_l2(f2.cpu().numpy(), field.cpu().numpy()) <= 1e-5
    near = Geometry(256, 256, 300.0, 1e5, K_UM, nf=True)
    hn = make_handle(lib, near, lib.PREC_FP32SPLIT)
    hn.forward(torch.from_numpy(atoms_ball(rng, 8192, 0.05)).cuda(), None, None, lib.OUT_INTENSITY, 0.05)
    assert hn.plan()["tile"] < 16
    zero = np.zeros((8192, 4))
    out = h.forward(torch.from_numpy(zero).cuda()).abs().cpu().numpy()
    np.testing.assert_allclose(out, 8192.0, rtol=1e-6)

