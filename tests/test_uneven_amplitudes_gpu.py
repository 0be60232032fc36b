"""Emitters and pixels far weaker than the brightest one keep their digits in the kernels that multiply FP16 pairs.

A kernel that scales by the largest of its range and splits into two FP16 parts has an absolute error of
FP16's smallest step; it has to lie below what FP32 leaves of every weaker emitter (or pixel).
"""
import numpy as np
import pytest

from conftest import K_UM
from gpu_util import atoms_ball, fp64_tol, make_handle, rel_l2, run

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    import torch

    from idi_amd import _lib

    assert torch.cuda.is_available()
    _lib.load()
    return _lib


def _geometry(shape):
    from oracle import Geometry

    return Geometry(*shape, 75.0, 2e5, K_UM, nf=True)


def _phasors(g, at):
    """e^{i theta} (pixels, emitters) in complex128 on the GPU, without the cancellation of D - z: the oracle's
    literal formula rounds a phase by up to fp64_tol (7e-6 here), more than the tolerances below."""
    import torch

    i, j = torch.meshgrid(torch.arange(g.n0, dtype=torch.float64), torch.arange(g.n1, dtype=torch.float64), indexing="ij")
    p = torch.stack([(i - g.n0 / 2) * g.pixelsize, (j - g.n1 / 2) * g.pixelsize, torch.full_like(i, g.detz)],
                    -1).reshape(-1, 3).cuda()
    e = torch.from_numpy(at).cuda()
    R = torch.linalg.vector_norm(p, dim=1, keepdim=True)
    t = (e[:, :3] ** 2).sum(1) - 2.0 * (p @ e[:, :3].T)
    th = g.k * (t / (torch.sqrt(R * R + t) + R) + e[:, 2] + (p[:, :1] ** 2 + p[:, 1:2] ** 2) / (R + p[:, 2:])) + e[:, 3]
    return torch.polar(torch.ones_like(th), th)


def _field(oracle_mod, g, at, amp):
    """The field in 64 bits, held to the oracle's within the latter's rounding."""
    ref = (_phasors(g, at).real @ _cuda(amp) + 1j * (_phasors(g, at).imag @ _cuda(amp))).cpu().numpy().reshape(g.n0, g.n1)
    assert rel_l2(oracle_mod.field_c(g, at, amp), ref) <= fp64_tol(g)
    return ref


def _cuda(a):
    import torch

    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _outlier(rng, n, ratio):
    """n emitters of amplitude 1 around one of amplitude `ratio` at the origin."""
    at = atoms_ball(rng, n, 0.01)
    at[n // 2, :3] = 0.0
    amp = np.ones(n)
    amp[n // 2] = ratio
    return at, amp


# The outlier's own phase is one rounded number in every pixel (2^-25 rev, 1.9e-7 rad) and its phasor one FP32
# sine (2^-22); a merge rounds its sum to 2^-24.  The others' errors, 1e-6 of each as a root mean square, add
# up to 1e-6 sqrt(n) / ratio, 2.4e-7 at most here.  Together below 1e-6; one part in 2^25 of the
# outlier in every emitter would be 3e-8 sqrt(20000) = 4e-6.
@pytest.mark.parametrize("tile", range(17, 23))
@pytest.mark.parametrize("ratio", [600.0, 1e5])
def test_weak_emitters_beside_a_bright_one(lib, oracle_mod, tile, ratio):
    g = _geometry((64, 96))
    at, amp = _outlier(np.random.default_rng(80), 20000, ratio)
    f, h = run(lib, g, at, amp, tile=tile, split=1)
    assert h.plan()["tile"] == tile
    assert np.isfinite(h.plan()["phase_bound"])
    assert rel_l2(f, _field(oracle_mod, g, at, amp)) <= 1e-6


def test_weak_emitters_of_a_batch(lib, oracle_mod):
    g = _geometry((64, 96))
    shots = [_outlier(np.random.default_rng(81 + s), 20000, 600.0) for s in range(2)]
    h = make_handle(lib, g, lib.PREC_FP32SPLIT)
    e, a = _cuda(np.concatenate([s[0] for s in shots])), _cuda(np.concatenate([s[1] for s in shots]))
    f = h.forward_batched(e, np.array([0, 20000, 40000]), a).cpu().numpy()
    assert 17 <= h.plan()["tile"] <= 22
    for i, (at, amp) in enumerate(shots):
        assert rel_l2(f[i], _field(oracle_mod, g, at, amp)) <= 1e-6


# The phases of a square's rows and columns take three roundings each, of numbers below 2 rev: as a root
# mean square sqrt(6) 2^-24 / sqrt(3) rev, 5e-7 rad where they are that large (the detector's edge).  FP32
# weights add 2^-25 of their own each.  Weights of 1e-3 that are split beside one of 1 in [1/2, 1) add
# sqrt(T^2) 2^-25 of that one besides: 4.8e-7 (T = 16) and 9.5e-7 (T = 32).
@pytest.mark.parametrize("shape,n,tile", [((64, 64), 3000, 22), ((256, 256), 20000, 18)])
def test_weak_pixels_beside_a_bright_one(lib, oracle_mod, shape, n, tile):
    rng = np.random.default_rng(83)
    g = _geometry(shape)
    at = atoms_ball(rng, n, 0.01)
    w = rng.normal(0, 1, shape)
    w *= 1e-3
    w[5::16, 9::16] *= 1e3
    w = w.astype(np.float32)
    f32 = (rng.normal(size=shape) + 1j * rng.normal(size=shape)).astype(np.complex64)
    h = make_handle(lib, g, lib.PREC_FP32SPLIT)
    gpos, gph, gamp = h.adjoint(_cuda(at), _cuda(f32), _cuda(w), None, 0.01 * (1 + 1e-9))
    assert h.plan()["tile"] == tile
    sub = np.arange(0, n, n // 300)
    # L = sum w |E|^2: d/d phase = 2 sum w Re(conj(E) i e^{i theta}), d/d amplitude without the i
    z = _phasors(g, at[sub])
    c = 2.0 * _cuda((w.astype(np.float64) * f32.astype(np.complex128).conj()).reshape(-1))
    ramp = (c.real @ z.real - c.imag @ z.imag).cpu().numpy()
    rph = -(c.real @ z.imag + c.imag @ z.real).cpu().numpy()
    _, oph, oamp = oracle_mod.adjoint_c(g, at[sub], w.astype(np.float64), field=f32.astype(np.complex128))
    assert rel_l2(oph, rph) <= fp64_tol(g) and rel_l2(oamp, ramp) <= fp64_tol(g)
    assert rel_l2(gph.cpu().numpy()[sub], rph) <= 5e-7
    assert rel_l2(gamp.cpu().numpy()[sub], ramp) <= 5e-7
