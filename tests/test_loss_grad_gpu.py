"""idisim_loss_grad_l2 against idisim_forward and idisim_adjoint_l2 where the forward takes the separable tiles."""
import numpy as np
import pytest

from conftest import K_UM
from gpu_util import atoms_ball, make_handle

pytestmark = pytest.mark.gpu

SEPARABLE = range(17, 23)


@pytest.mark.parametrize("shape,n,amp,opts", [
    ((256, 256), 8192, False, {}),                       # the fit workload's detector, 5.4e8 pairs
    ((512, 512), 2048, True, {}),
    ((333, 211), 16400, True, {}),                       # ragged
    ((256, 256), 8192, False, {"autotune": 0}),
    ((256, 256), 8192, True, {"split": 1}),              # no partials: the forward finalizes on its own
    ((64, 48), 600, True, {"tile": 17}),
    ((64, 48), 600, False, {"tile": 22, "split": 2}),
])
def test_the_same_bits_in_one_call(shape, n, amp, opts):
    import torch

    from idi_amd import _lib as lib
    from oracle import Geometry

    rng = np.random.default_rng(97)
    g = Geometry(*shape, 75.0, 2e5, K_UM, nf=True)
    at = atoms_ball(rng, n, 0.01)
    h = make_handle(lib, g, lib.PREC_FP32SPLIT)
    for k, v in opts.items():
        h.set_option(getattr(lib, "OPT_" + k.upper()), v)
    d = torch.from_numpy(at).cuda()
    a = torch.from_numpy(rng.uniform(0.5, 1, n)).cuda() if amp else None
    T = torch.from_numpy((rng.exponential(n, shape)).astype(np.float32)).cuda()
    ext = float(np.linalg.norm(at[:, :3], axis=1).max())
    field = h.forward(d, a, None, lib.OUT_FIELD, ext)
    assert h.plan()["tile"] in SEPARABLE
    ref = h.adjoint_l2(d, field, T, a, ext, want_amp=amp)
    f2 = torch.full_like(field, float("nan"))
    for out in (f2, None):  # with and without the field output
        got = h.loss_grad_l2(d, T, a, ext, field=out, want_amp=amp)
        assert got[0].item() == ref[0].item()
        for x, y in zip(got[1:], ref[1:]):
            assert y is None or torch.equal(x, y)
    assert torch.equal(f2, field)
