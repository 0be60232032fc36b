"""Long sums on the matrix cores have no bias.

A matrix instruction truncates its sums of eight products downwards, 7e-10 per emitter of amplitude 1 in the
real and the imaginary part alike: nothing in one image of few emitters, but it grows with their number
where a sum of random phases grows with its square root.
"""
import numpy as np
import pytest

from conftest import K_UM
from gpu_util import atoms_ball, make_handle, rel_l2, run
from test_uneven_amplitudes_gpu import _cuda, _phasors

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    import torch

    from idi_amd import _lib

    assert torch.cuda.is_available()
    _lib.load()
    return _lib


# Far field (no phase of the pixel's own, and the oracle exact to 1e-9).  The speckles of a 50 nm ball are 15 pixels wide, so
# 256 x 256 pixels hold about 290 independent errors, whose mean is 1/17 of their root mean square; a quarter
# is 4 standard deviations.  7e-10 (1 + i) for each of 300000 emitters is 5.5e-4, against errors of
# 4e-7 sqrt(300000) = 2.2e-4 each.
@pytest.mark.parametrize("tile", range(17, 23))
@pytest.mark.parametrize("split,amplitudes", [(1, False), (1, True), (5, False)])
def test_forward(lib, oracle_mod, tile, split, amplitudes):
    from oracle import Geometry

    rng = np.random.default_rng(130)
    g = Geometry(256, 256, 50.0, 5e5, K_UM)
    n = 300000
    at = atoms_ball(rng, n, 0.05)
    amp = rng.uniform(0.9, 1.1, n) if amplitudes else None
    rows = np.arange(5, 256, 16)
    f, h = run(lib, g, at, amp, tile=tile, split=split)
    assert h.plan()["tile"] == tile and h.plan()["phase_bound"] <= 5e-6
    d = f[rows] - oracle_mod.field_c(g, at, amp, rows=[int(r) for r in rows])
    assert abs(d.mean()) <= np.sqrt((np.abs(d) ** 2).mean()) / 4


# Three roundings each of the phases of a square's rows and columns, of numbers below 2 rev: 5e-7 rad as a root
# mean square where they are that large (as in test_weak_pixels_beside_a_bright_one).
@pytest.mark.parametrize("side,pix,z,tile", [(2000, 50.0, 5e5, 18), (1500, 100.0, 2.5e5, 22)])
def test_adjoint(lib, side, pix, z, tile):
    from oracle import Geometry

    rng = np.random.default_rng(131)
    g = Geometry(side, side, pix, z, K_UM, nf=True)
    at = atoms_ball(rng, 400, 0.03)
    w = rng.normal(size=(side, side)).astype(np.float32)
    f = (rng.normal(size=w.shape) + 1j * rng.normal(size=w.shape)).astype(np.complex64)
    h = make_handle(lib, g, lib.PREC_FP32SPLIT)
    _, gph, gamp = h.adjoint(_cuda(at), _cuda(f), _cuda(w), None, 0.03 * (1 + 1e-9))
    assert h.plan()["tile"] == tile
    c = 2.0 * _cuda((w.astype(np.float64) * f.astype(np.complex128).conj()).reshape(-1))
    rph, ramp = np.empty(400), np.empty(400)
    for i in range(0, 400, 50):
        z_ = _phasors(g, at[i:i + 50])
        ramp[i:i + 50] = (c.real @ z_.real - c.imag @ z_.imag).cpu().numpy()
        rph[i:i + 50] = -(c.real @ z_.imag + c.imag @ z_.real).cpu().numpy()
    assert rel_l2(gph.cpu().numpy(), rph) <= 5e-7
    assert rel_l2(gamp.cpu().numpy(), ramp) <= 5e-7
