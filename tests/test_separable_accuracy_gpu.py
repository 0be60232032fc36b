"""The separable forward tiles to the digits that they claim: both FP16 parts, the mixed remainder's terms, and
every variant in every phase model at a distance where the planner would take it."""
import numpy as np
import pytest

from conftest import K_UM
from gpu_util import atoms_ball, fp64_tol, make_handle, rel_l2, run
from test_uneven_amplitudes_gpu import _phasors

pytestmark = pytest.mark.gpu

TILES = range(17, 23)


@pytest.fixture(scope="module")
def lib():
    import torch

    from idi_amd import _lib

    assert torch.cuda.is_available()
    _lib.load()
    return _lib


def _exact(g, at, amp=None):
    """The field in 64 bits without the cancellation of the literal near-field formula."""
    z = _phasors(g, at)
    f = z.sum(1) if amp is None else z @ z.new_tensor(amp)
    return f.cpu().numpy().reshape(g.n0, g.n1)


def _rms_tol(plan):
    """Relative L2 of many emitters with random phases: the terms' errors add as root mean squares.  The
    phase bound is a sum of ten and more worst cases (roundings, each at most 1 / sqrt(3) of its largest as a
    root mean square, and a remainder that is reached at the corners alone): a quarter of it.  2^-21 for the
    sines (2^-22), the two FP16 parts of both phasors (2^-23 each) and the FP32 sums.  One lost low part is
    1.7e-4."""
    assert np.isfinite(plan["phase_bound"]) and plan["phase_bound"] <= 5e-6, plan
    return 2 * np.pi * plan["phase_bound"] / 4 + 2.0**-21


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("amplitudes", [False, True])
def test_many_random_emitters(lib, tile, amplitudes):
    from oracle import Geometry

    rng = np.random.default_rng(110)
    g = Geometry(90, 150, 75.0, 4e5, K_UM, nf=True)
    at = atoms_ball(rng, 8000, 0.01)
    amp = rng.uniform(0.5, 1.0, 8000) if amplitudes else None
    for split in (1, 8):
        f, h = run(lib, g, at, amp, tile=tile, split=split)
        assert h.plan()["tile"] == tile
        tol = _rms_tol(h.plan())
        assert tol <= 5e-6
        assert rel_l2(f, _exact(g, at, amp)) <= tol


# 100 um pixels at 0.1 m with emitters up to 30 nm off: the mixed phase M reaches 1.2e-2 rad over 16 x 16 pixels
# and only tile 22 meets the bound; its second-order term M^2 / 2 is 7.2e-5 there.
def _coarse():
    from oracle import Geometry

    return Geometry(256, 256, 100.0, 1e5, K_UM, nf=True)


@pytest.mark.parametrize("direction", [(1, 1, 0), (1, -1, 0), (1, 1, 1), (0, 1, 0), (0, 0, 1)])
def test_second_order_of_one_emitter(lib, direction):
    """One emitter at the extent, in every pixel: within the phase bound (2.3e-5 rad), which the second-order
    term exceeds three times; 2^-21 as in _rms_tol.  The amplitude is 1 in every pixel."""
    g = _coarse()
    at = np.zeros((1, 4))
    at[0, :3] = 0.03 * np.array(direction) / np.linalg.norm(direction)
    at[0, 3] = 0.7
    h = make_handle(lib, g, lib.PREC_FP32SPLIT)
    f, h = run(lib, g, at, tile=22, split=1, handle=h)
    p = h.plan()
    assert p["tile"] == 22 and p["phase_bound"] <= 5e-6
    err = np.abs(f - _exact(g, at)).max()
    tol = 2 * np.pi * p["phase_bound"] + 2.0**-21
    assert tol <= 3e-5
    assert err <= tol, (err, tol)


@pytest.mark.parametrize("amplitudes", [False, True])
def test_second_order_of_an_image(lib, amplitudes):
    import torch

    g = _coarse()
    rng = np.random.default_rng(112)
    n = 2000
    at = [atoms_ball(rng, n, 0.03) for _ in range(2)]
    amp = [rng.uniform(0.5, 1.0, n) for _ in range(2)]
    h = make_handle(lib, g, lib.PREC_FP32SPLIT)
    e = torch.from_numpy(np.concatenate(at)).cuda()
    a = torch.from_numpy(np.concatenate(amp)).cuda() if amplitudes else None
    f = h.forward_batched(e, np.array([0, n, 2 * n]), a, extent=0.03).cpu().numpy()
    assert h.plan()["tile"] == 22  # chosen: no other separable tile meets the bound
    for s in range(2):
        assert rel_l2(f[s], _exact(g, at[s], amp[s] if amplitudes else None)) <= _rms_tol(h.plan())


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("mode", ["nf", "nf scale amp", "ff", "ff secondorder", "ff scale amp", "nf rot"])
def test_phase_models_where_the_tile_is_taken(lib, oracle_mod, tile, mode):
    """Per pixel: the planner's phase bound for every term, the FP32 roundings of the sums (at most 192 matrix
    instructions between two merges) and the oracle's own rounding."""
    from oracle import Geometry

    rng = np.random.default_rng(113)
    rot = "rot" in mode
    z = 6e5
    g = Geometry(70, 135, 75.0, z, K_UM, detoffset=(900.0, -1500.0) if rot else (0.0, 0.0),
                 detangles=(0.05, -0.08) if rot else (0.0, 0.0), nf=mode.startswith("nf"), scale="scale" in mode,
                 secondorder="secondorder" in mode)
    at = atoms_ball(rng, 700, 0.01)
    amp = rng.uniform(0.5, 1.0, 700) if "amp" in mode else None
    f, h = run(lib, g, at, amp, tile=tile, split=2)
    p = h.plan()
    assert p["tile"] == tile and p["phase_bound"] <= 5e-6  # finite: the planner would take it
    total = (700 if amp is None else amp.sum()) / (z if g.scale else 1.0)
    tol = (2 * np.pi * p["phase_bound"] + 192 * 2.0**-24 + fp64_tol(g)) * total
    assert np.abs(f - oracle_mod.field_c(g, at, amp)).max() <= tol
