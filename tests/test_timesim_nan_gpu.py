"""A NaN arrival time (which leaves the sort behind the padding) gives NaN pixels
where one workgroup takes a pixel."""
import numpy as np
import pytest

from conftest import K_UM
from gpu_util import atoms_ball, make_handle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [False, True])
@pytest.mark.parametrize("n,where", [(1, 0), (10, 9), (1024, 0), (1025, 500), (9000, 8999)])
def test_nan_time(n, where, scale):
    import torch

    from idi_amd import _lib as lib
    from oracle import Geometry

    rng = np.random.default_rng(120)
    g = Geometry(5, 3, 300.0, 1e5, K_UM, nf=True, scale=scale)
    e = torch.from_numpy(atoms_ball(rng, n, 0.02)).cuda()
    t = torch.from_numpy(5e-4 * rng.normal(size=n)).cuda()
    for precision in (lib.PREC_FP32SPLIT, lib.PREC_FP64):
        h = make_handle(lib, g, precision)
        h.set_option(lib.OPT_TIME_PATH, 1)
        good = h.time_forward(e, t, 0.299792458, 1e-3)
        assert torch.isfinite(good).all()
        bad = t.clone()
        bad[where] = float("nan")
        assert torch.isnan(h.time_forward(e, bad, 0.299792458, 1e-3)).all(), precision
        assert torch.equal(h.time_forward(e, t, 0.299792458, 1e-3), good)
