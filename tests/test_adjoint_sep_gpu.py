"""The separable adjoint (matrix products over the pixels) against the FP64 analytic gradient of the oracle."""
import numpy as np
import pytest

from conftest import K_UM
from gpu_util import atoms_ball, ball, fp64_tol, make_handle, rel_l2

pytestmark = pytest.mark.gpu

SIDE32, SIDE16, PER_PIXEL = 18, 22, 0  # the tile that the plan reports
MODES = ["nf", "nf scale amp", "ff", "ff secondorder amp", "nf rot"]


@pytest.fixture(scope="module")
def lib():
    import torch

    from idi_amd import _lib

    assert torch.cuda.is_available()
    _lib.load()
    return _lib


def _geometry(shape, mode, pix=75.0, z=2e5):
    from oracle import Geometry

    rot = "rot" in mode
    return Geometry(*shape, pix, z, K_UM, detoffset=(900.0, -1500.0) if rot else (0.0, 0.0),
                    detangles=(0.05, -0.08) if rot else (0.0, 0.0), nf=mode.startswith("nf"), scale="scale" in mode,
                    secondorder="secondorder" in mode)


def _check(lib, oracle_mod, g, mode, n, seed, tile, weights=None):
    """Per emitter, the planner's phase bound for every pair and the FP32 roundings of the sums (two FP16
    parts, 64 additions) of its phase and amplitude gradients; the position gradient as in the tests of the
    per-pixel kernel."""
    import torch

    rng = np.random.default_rng(seed)
    at = atoms_ball(rng, n, 0.01)
    amp = rng.uniform(0.5, 1.0, n) if "amp" in mode else None
    f32 = oracle_mod.field_c(g, at, amp).astype(np.complex64)
    w = rng.normal(0, 1, f32.shape).astype(np.float32)
    if weights is not None:
        w *= weights(w.shape)
    rpos, rph, ramp = oracle_mod.adjoint_c(g, at, w.astype(np.float64), field=f32.astype(np.complex128), amp=amp)
    h = make_handle(lib, g, lib.PREC_FP32SPLIT)
    d = torch.from_numpy(at).cuda()
    da = None if amp is None else torch.from_numpy(amp).cuda()
    ext = 0.01 * (1 + 1e-9)
    args = (torch.from_numpy(f32).cuda(), torch.from_numpy(w).cuda(), da, ext)
    gpos, gph, gamp = h.adjoint(d, *args)
    qpos, qph, none = h.adjoint(d, *args, want_amp=False)
    p = h.plan()
    assert p["tile"] == tile and p["phase_bound"] <= 5e-6, p
    assert none is None and torch.equal(qpos, gpos) and torch.equal(qph, gph)
    total = 2 * np.abs(w.astype(np.float64) * f32).sum() / (g.detz if g.scale else 1.0)
    tol = (2 * np.pi * p["phase_bound"] + 2.0**-22 + 64 * 2.0**-24 + fp64_tol(g)) * total
    assert np.abs(gph.cpu().numpy() - rph).max() <= tol
    assert np.abs(gamp.cpu().numpy() - ramp).max() <= tol
    if n > 1:  # one pixel's intensity of one emitter does not depend on its position
        assert rel_l2(gpos.cpu().numpy().astype(np.float64), rpos) <= 2e-5


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("shape,n,tile", [((1, 1), 1, SIDE16), ((16, 33), 17, SIDE16), ((31, 47), 257, SIDE16),
                                          ((65, 80), 1030, SIDE16), ((1, 2049), 8200, SIDE16),
                                          ((33, 1025), 15700, SIDE32), ((65, 129), 43777, SIDE32)])
def test_edges_of_squares_and_groups(lib, oracle_mod, shape, n, tile, mode):
    """Detectors at and one past the edges of the squares and of the 2 x 2 squares of a workgroup; emitters
    at and around a step and a group of 256; enough workgroups for squares of 32 pixels or not."""
    _check(lib, oracle_mod, _geometry(shape, mode), mode, n, 60 + n, tile)


def test_weights_over_many_decades(lib, oracle_mod):
    """Weights that differ by nine decades from square to square (each has its own scale), and empty squares."""
    def weights(shape):
        s = 10.0 ** (3 * ((np.arange(shape[0])[:, None] // 16 + np.arange(shape[1])[None] // 16) % 4) - 6)
        s[16:32] = 0.0
        return s.astype(np.float32)

    _check(lib, oracle_mod, _geometry((64, 100), "nf"), "nf", 500, 61, SIDE16, weights)


def test_coarse_geometry_keeps_the_per_pixel_kernel(lib, oracle_mod):
    """300 um pixels at 0.1 m: the mixed terms over 16 pixels are too large."""
    import torch

    rng = np.random.default_rng(62)
    g = _geometry((64, 48), "nf", 300.0, 1e5)
    at = np.concatenate([ball(rng, 300, 0.02), rng.uniform(0, 2 * np.pi, (300, 1))], 1)
    h = make_handle(lib, g, lib.PREC_FP32SPLIT)
    d = torch.from_numpy(at).cuda()
    field = h.forward(d)
    h.adjoint(d, field, torch.ones((64, 48), device="cuda"), None, 0.0200001)
    assert h.plan()["tile"] == PER_PIXEL
