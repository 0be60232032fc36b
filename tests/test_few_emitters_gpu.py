"""Many pixels and few emitters a shot: the separable tiles, which pay per rectangle, are not taken by the number
of pairs alone."""
import numpy as np
import pytest

from conftest import K_UM
from gpu_util import atoms_ball, make_handle, rel_l2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    import torch

    from idi_amd import _lib

    assert torch.cuda.is_available()
    _lib.load()
    return _lib


def _handle(lib, side, coarse, autotune=0):
    """coarse: the 16 x 16 rectangles alone meet the bound."""
    from oracle import Geometry

    g = Geometry(side, side, 100.0, 1e5 if side < 1000 else 2.5e5, K_UM, nf=True) if coarse else \
        Geometry(side, side, 75.0, 3e5, K_UM, nf=True)
    h = make_handle(lib, g, lib.PREC_FP32SPLIT)
    h.set_option(lib.OPT_AUTOTUNE, autotune)
    return g, h


# without timing: the separable tiles from 96 emitters on, never below 32 also where candidates are timed
@pytest.mark.parametrize("coarse", [False, True])
@pytest.mark.parametrize("autotune", [0, 1])
@pytest.mark.parametrize("n,shots", [(4, 400), (31, 60), (40, 50), (95, 20), (96, 20), (130, 14)])
def test_batches_of_small_shots(lib, oracle_mod, coarse, autotune, n, shots):
    import torch

    g, h = _handle(lib, 256, coarse, autotune)
    r = 0.03 if coarse else 0.01
    rng = np.random.default_rng(90 + n)
    at = [atoms_ball(rng, n, r) for _ in range(shots)]
    offs = np.arange(shots + 1, dtype=np.int64) * n
    assert offs[-1] * 256 * 256 >= 1e8
    e = torch.from_numpy(np.concatenate(at)).cuda()
    out = h.forward_batched(e, offs, None, None, lib.OUT_INTENSITY, r).cpu().numpy()
    tile = h.plan()["tile"]
    if n < 32 or (not autotune and n < 96):
        assert tile < 16
    elif n >= 128 or not autotune:
        assert tile >= 17
    assert rel_l2(out[shots - 1], np.abs(oracle_mod.field_c(g, at[-1])) ** 2) <= 1e-4


@pytest.mark.parametrize("coarse", [False, True])
@pytest.mark.parametrize("autotune", [0, 1])
@pytest.mark.parametrize("n", [31, 33, 95, 96, 130])
def test_few_emitters_on_a_large_detector(lib, oracle_mod, coarse, autotune, n):
    import torch

    g, h = _handle(lib, 2000, coarse, autotune)
    r = 0.03 if coarse else 0.01
    at = atoms_ball(np.random.default_rng(91), n, r)
    e = torch.from_numpy(at).cuda()
    for _ in range(2):  # chosen, and from the plan's cache
        out = h.forward(e, None, None, lib.OUT_INTENSITY, r)
        tile = h.plan()["tile"]
        if n < 32 or (not autotune and n < 96):
            assert tile < 16
        elif n >= 128 or not autotune:
            assert tile >= 17
    rows = [0, 999, 1999]
    ref = np.abs(oracle_mod.field_c(g, at, rows=rows)) ** 2
    assert rel_l2(out.cpu().numpy()[rows], ref) <= 1e-4
