"""The work that users of this framework have it do, as cases that can be timed.

listed()          the cases: each a dict of plain values with a name
draw(rng)         one more case of the same ranges
prepare(case, s)  the inputs of a case (from the seed s alone) and the handle that a program keeps
run(state)        one pass through the public entry points
work(case)        the bytes and operations that a pass cannot do without
exact(case, s)    the same outputs in 64 bits with plain torch

Lengths are in micrometres and k in rad per micrometre (0.154 nm X-rays), as in the rest of the repository.
"""
import math

import numpy as np
import torch

from idi_amd import _lib
from idi_amd.reconstruction import qcor
from idi_amd.simulation import autograd, common, hip

K = 2 * math.pi / 1.54e-4
BALLS = ((-0.040, 0.015), (0.0, 0.020), (0.050, 0.025))  # (x of the centre, radius): three balls 5 nm apart


def listed():
    return [
        # the smallest image: a first try of a geometry, or one image of a long loop over random phases;
        # a thousand emitters, where the launches and the host path count
        dict(name="image_small", kind="image", n0=128, n1=128, n=1000, pix=75.0, z=1e5, shape="ball", r=0.05,
             settings="single nf", intensity=False, amp=False),
        # the same in double precision, the default of simulate()
        dict(name="image_small_double", kind="image", n0=128, n1=128, n=1000, pix=75.0, z=1e5, shape="ball", r=0.05,
             settings="double nf", intensity=False, amp=False),
        # the ordinary image: a 10 nm simple-cubic nanocrystal on a 512 x 512 detector
        dict(name="image_crystal", kind="image", n0=512, n1=512, n=100000, pix=75.0, z=2e5, shape="lattice", r=0.01,
             settings="single nf", intensity=False, amp=False),
        # a double-precision image of middle size (a reference run, or a geometry too close for "single")
        dict(name="image_double", kind="image", n0=256, n1=256, n=20000, pix=75.0, z=1e5, shape="ball", r=0.02,
             settings="double nf", intensity=False, amp=False),
        # far field with the options set: an odd, ragged, rotated and shifted detector, 1/r amplitudes, the
        # second-order phase, per-emitter amplitudes, intensity output
        dict(name="image_far_ragged", kind="image", n0=333, n1=211, n=12345, pix=55.0, z=1.5e5, shape="ball", r=0.02,
             settings="single scale secondorder", intensity=True, amp=True, angles=True),
        # many shots of a jet or a rastered target: uneven emitter counts, fresh phases, one call
        dict(name="shots_batched", kind="shots", n0=256, n1=256, nshots=64, nlo=1000, nhi=50000, pix=100.0, z=1e5,
             shape="ball", r=0.03, settings="single nf", intensity=True, amp=False),
        # the largest: a million emitters with amplitudes in three balls, megapixel images, two shots
        dict(name="shots_large", kind="shots", n0=1024, n1=1024, nshots=2, nlo=1000000, nhi=1000000, pix=50.0, z=5e5,
             shape="balls", r=0.075, settings="single nf", intensity=False, amp=True),
        # one step of a fit of positions and phases to a measured intensity
        dict(name="fit_step", kind="fit", n0=256, n1=256, n=4096, pix=75.0, z=1e5, shape="ball", r=0.02,
             settings="single nf"),
        # forward and backward of the differentiable intensity under another loss, with amplitudes, larger
        dict(name="intensity_grad", kind="grad", n0=512, n1=512, n=20000, pix=75.0, z=2e5, shape="ball", r=0.02,
             settings="single nf", amp=True),
        # time-dependent image of decaying emitters (float32 arrival times)
        dict(name="time_image", kind="time", n0=128, n1=128, n=10000, pix=300.0, z=1e5, shape="ball", r=0.02,
             settings="single nf"),
        # photon counting and charge sharing of a simulated intensity image
        dict(name="photons", kind="photons", n0=512, n1=512, photons=1e6, sigma=0.75, gain=0.1),
        # q-corrected correlation of one photon image, to the host as its call returns it
        dict(name="q_correlation", kind="qcorr", n0=256, n1=256, z=2000.0, maxq=64, mean=2.0),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _side(rng, lo, hi):
    return int(round(_log(rng, lo, hi)))


def draw(rng):
    kind = rng.choice(["image"] * 5 + ["shots"] * 2 + ["fit", "grad", "time", "photons", "qcorr"])
    if kind == "photons":
        return dict(kind=kind, n0=_side(rng, 100, 900), n1=_side(rng, 100, 900), photons=float(round(_log(rng, 1e4, 3e6))),
                    sigma=rng.uniform(0.3, 1.6), gain=rng.choice([0.0, 0.1]))
    if kind == "qcorr":
        return dict(kind=kind, n0=_side(rng, 100, 400), n1=_side(rng, 100, 400), z=rng.uniform(1000, 4000),
                    maxq=rng.randint(32, 96), mean=rng.uniform(0.2, 4.0))
    near = rng.random() < 0.75
    c = dict(kind=kind, pix=rng.uniform(40, 110), z=_log(rng, 1e5, 6e5), r=_log(rng, 0.008, 0.06), shape="ball")
    if kind == "time":
        return dict(c, n0=_side(rng, 40, 160), n1=_side(rng, 40, 160), n=_side(rng, 500, 20000), pix=300.0,
                    settings=rng.choice(["single", "double"]) + (" nf" if near else ""))
    if kind in ("fit", "grad"):
        return dict(c, n0=_side(rng, 100, 600), n1=_side(rng, 100, 600), n=_side(rng, 1000, 30000),
                    settings="single" + (" nf" if near else ""), amp=kind == "grad" and rng.random() < 0.5)
    single = kind == "shots" or rng.random() < 0.75
    c.update(intensity=rng.random() < 0.5, amp=rng.random() < 0.4,
             settings=("single" if single else "double") + (" nf" if near else rng.choice(["", " secondorder"])) +
             rng.choice(["", "", " scale"]))
    if kind == "shots":
        hi = _side(rng, 500, 60000)
        return dict(c, n0=_side(rng, 60, 400), n1=_side(rng, 60, 400), nshots=rng.randint(2, 40), nlo=max(1, hi // 20),
                    nhi=hi)
    big = 100000 if single else 20000
    return dict(c, n0=_side(rng, 60, 700), n1=_side(rng, 60, 700), n=_side(rng, 300, big), angles=rng.random() < 0.3,
                shape=rng.choice(["ball", "ball", "lattice"]))


# ------------------------------------------------------------------------------ inputs


def _ball(gen, n, r):
    v = torch.randn((n, 3), generator=gen, dtype=torch.float64, device="cuda")
    v /= torch.linalg.vector_norm(v, dim=1, keepdim=True)
    return v * r * torch.rand((n, 1), generator=gen, dtype=torch.float64, device="cuda") ** (1 / 3)


def _emitters(case, gen, n):
    """(n, 4) float64 emitters (x, y, z, phase) of the case's object."""
    e = torch.empty((n, 4), dtype=torch.float64, device="cuda")
    r = case["r"]
    if case["shape"] == "lattice":  # n of the 1.55 n simple-cubic sites in the ball (0.3 nm apart for 100000 in 10 nm)
        a = r * (4 * math.pi / 3 / (1.55 * n)) ** (1 / 3)
        m = int(math.ceil(r / a))
        g = torch.arange(-m, m + 1, dtype=torch.float64, device="cuda") * a
        pts = torch.stack(torch.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
        pts = pts[torch.linalg.vector_norm(pts, dim=1) <= r]
        e[:, :3] = pts[torch.randperm(len(pts), generator=gen, device="cuda")[:n]]
    elif case["shape"] == "balls":
        vol = np.array([b[1] ** 3 for b in BALLS])
        cnt = np.rint(n * vol / vol.sum()).astype(int)
        cnt[-1] = n - cnt[:-1].sum()
        parts = []
        for (x, rb), k in zip(BALLS, cnt):
            p = _ball(gen, int(k), rb)
            p[:, 0] += x
            parts.append(p)
        e[:, :3] = torch.cat(parts)
    else:
        e[:, :3] = _ball(gen, n, r)
    e[:, 3] = torch.rand(n, generator=gen, dtype=torch.float64, device="cuda") * (2 * math.pi)
    return e


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) % (1 << 62))
    return g


def _detector(case):
    """(detangles, detoffset): tilted by a few degrees and shifted, or centred."""
    return ((0.03, 0.1), (900.0, -650.0)) if case.get("angles") else ((0, 0), (0, 0))


def _counts(case, seed):
    rng = np.random.default_rng(seed)
    return rng.integers(case["nlo"], case["nhi"] + 1, case["nshots"])


def _inputs(case, seed):
    """The case's tensors by name: the same for run() and exact()."""
    g, kind = _gen(seed), case["kind"]
    shape = (case["n0"], case["n1"])
    f64 = dict(generator=g, dtype=torch.float64, device="cuda")
    if kind == "photons":  # speckle: exponential intensities
        return {"image": -torch.log(1 - torch.rand(shape, **f64))}
    if kind == "qcorr":
        lam = torch.full(shape, case["mean"], dtype=torch.float32, device="cuda")
        return {"image": torch.poisson(lam, generator=g)}
    if kind == "shots":
        n = _counts(case, seed)
        x = {"emit": _emitters(case, g, int(n.sum())), "offsets": np.concatenate([[0], np.cumsum(n)]).astype(np.int64)}
    else:
        x = {"emit": _emitters(case, g, case["n"])}
    if case.get("amp"):
        x["amp"] = 0.5 + 0.5 * torch.rand(len(x["emit"]), **f64)
    if kind == "time":
        x["times"] = 5e-4 * torch.randn(len(x["emit"]), **f64)
    if kind == "fit":  # the measured image: another phase draw of the same mean intensity
        x["target"] = (-torch.log(1 - torch.rand(shape, **f64)) * case["n"]).float()
    if kind == "grad":
        x["pos"], x["phase"] = x["emit"][:, :3].float(), x["emit"][:, 3].float()
        if "amp" in x:
            x["amp"] = x["amp"].float()
        x["up"] = torch.randn(shape, generator=g, dtype=torch.float32, device="cuda") / case["n"]
    return x


def prepare(case, seed):
    x = _inputs(case, seed)
    st = {"case": case, "x": x, "seed": int(seed) % (1 << 31)}
    if case["kind"] in ("photons", "qcorr"):
        if case["kind"] == "qcorr":
            st["ctx"] = qcor.corrfunction((case["n0"], case["n1"]), case["z"], case["maxq"])
            st["corr"] = st["ctx"].__enter__()
        return st
    angles, offset = _detector(case)
    st["geom"] = ((case["n0"], case["n1"]), case["pix"], case["z"], K)
    st["det"] = dict(settings=case["settings"], detangles=angles, detoffset=offset)
    st["extent"] = case["r"] * (1 + 1e-9)
    if case["kind"] == "grad":
        st["extent"] *= 1 + 1e-6  # float32 positions
        st["leaves"] = [x["pos"].requires_grad_(), x["phase"].requires_grad_()]
        if "amp" in x:
            st["leaves"].append(x["amp"].requires_grad_())
    else:
        st["handle"] = hip.get_handle(*st["geom"], **st["det"])
    return st


def run(st):
    case, x = st["case"], st["x"]
    kind = case["kind"]
    if kind == "image":
        out = _lib.OUT_INTENSITY if case["intensity"] else _lib.OUT_FIELD
        return st["handle"].forward(x["emit"], x.get("amp"), None, out, st["extent"])
    if kind == "shots":
        return hip.simulate_batched((x["emit"], x["offsets"]), *st["geom"], **st["det"], amplitudes=x.get("amp"),
                                    intensity=case["intensity"], returngpu=True, extent=st["extent"])
    if kind == "fit":
        loss, gpos, gphase, _ = st["handle"].loss_grad_l2(x["emit"], x["target"], None, st["extent"], want_amp=False)
        return {"loss": loss, "pos": gpos, "phase": gphase}
    if kind == "grad":
        inten = autograd.intensity(*st["leaves"], Ndet=st["geom"][0], pixelsize=case["pix"], detz=case["z"], k=K,
                                   **st["det"], extent=st["extent"])
        grads = torch.autograd.grad(inten, st["leaves"], x["up"])
        return {"intensity": inten.detach(), "grads": list(grads)}
    if kind == "time":
        return st["handle"].time_forward(x["emit"], x["times"], 0.299792458, 1e-3)
    if kind == "photons":
        counts = common.randomphotons(x["image"], case["photons"], rng=st["seed"])
        return {"counts": counts, "charge": common.chargesharing(counts, case["sigma"], case["gain"], rng=st["seed"] + 1)}
    return st["corr"](x["image"])


def _ewald(case):
    """(z / distance of every pixel in float32, the half width of the dqz bins) of a q-corrected correlation."""
    i, j = np.meshgrid(np.arange(case["n0"]) - case["n0"] / 2, np.arange(case["n1"]) - case["n1"] / 2, indexing="ij")
    zd = (case["z"] / np.sqrt(i * i + j * j + case["z"] ** 2)).astype(np.float32)
    return zd, int(math.ceil(case["z"] * float(zd.max() - zd.min()))) | 1


def work(case):
    """A direct sum needs one complex multiply-add (8 operations) per emitter and pixel; a gradient pass as much
    for the field's weight and for its three position moments; the decaying emitters an arrival time, an
    amplitude and a step of the scan (30); a q-corrected pair three bins and a multiply-add (12)."""
    p, kind = case["n0"] * case["n1"], case["kind"]
    if kind == "photons":
        w = 2 * int(math.ceil(2 * case["sigma"])) + 1
        return {"bytes": 3 * 8 * p, "flops": case["photons"] * (w * w * 3 + w * 60)}
    if kind == "qcorr":
        q = max(32, min(1024, case["maxq"], case["n0"], case["n1"]))
        rows = sum(case["n0"] - d for d in range(q))
        cols = sum(case["n1"] - abs(d) for d in range(1 - q, q))
        return {"bytes": 4 * p * 2 + 8 * 8 * _ewald(case)[1] * q * q, "flops": 12.0 * rows * cols}
    wide = 2 if "double" in case["settings"] else 1
    if kind == "shots":
        n = case["nshots"] * (case["nlo"] + case["nhi"]) / 2
        return {"bytes": n * (40 if case["amp"] else 32) + case["nshots"] * p * (4 if case["intensity"] else 8),
                "flops": 8.0 * n * p}
    n = case["n"]
    if kind == "time":
        return {"bytes": 40 * n + 8 * p, "flops": 30.0 * n * p}
    if kind == "image":
        return {"bytes": n * (40 if case["amp"] else 32) + p * (4 if case["intensity"] else 8) * wide, "flops": 8.0 * n * p}
    return {"bytes": 48 * n + 8 * p, "flops": 24.0 * n * p}


# ------------------------------------------------------------------------------ in 64 bits


def _rotation(alpha, beta):
    """Rotation by alpha about x, then by beta about y."""
    ca, sa, cb, sb = math.cos(alpha), math.sin(alpha), math.cos(beta), math.sin(beta)
    return np.array([[cb, sa * sb, ca * sb], [0.0, ca, -sa], [-sb, sa * cb, ca * cb]])


def _pixels(case):
    """Pixel positions (P, 3) in float64."""
    (theta, phi), (o0, o1) = _detector(case)
    i, j = torch.meshgrid(torch.arange(case["n0"], dtype=torch.float64, device="cuda"),
                          torch.arange(case["n1"], dtype=torch.float64, device="cuda"), indexing="ij")
    p = torch.stack([(i - case["n0"] / 2) * case["pix"] + o0, (j - case["n1"] / 2) * case["pix"] + o1,
                     torch.full_like(i, case["z"])], -1).reshape(-1, 3)
    if theta or phi:
        p = p @ torch.from_numpy(np.ascontiguousarray(_rotation(theta, phi).T)).cuda()
    return p


def _phases(case, p, e):
    """(phase, distance) of the emitters e at the pixels p, without the pixels' own k (R - z)."""
    R = torch.linalg.vector_norm(p, dim=1, keepdim=True)
    if " nf" not in case["settings"]:
        u = p / R
        u = torch.stack([u[:, 0], u[:, 1], -(p[:, 0] ** 2 + p[:, 1] ** 2) / (R[:, 0] * (R[:, 0] + p[:, 2]))], 1)
        th = torch.addmm(e[:, 3].expand(len(p), -1), u, e[:, :3].T, alpha=-K)
        if "secondorder" in case["settings"]:
            th += K / (2 * R) * (e[:, 0] ** 2 + e[:, 1] ** 2)
        return th, R
    t = torch.addmm((e[:, :3] ** 2).sum(1).expand(len(p), -1), p, e[:, :3].T, alpha=-2.0)
    D = (t + R * R).sqrt_()
    th = t.div_(D + R).mul_(K).add_(K * e[:, 2] + e[:, 3])
    return th, D


def _field(case, e, a, p):
    """E in complex128 at the pixels p, in slices of pixels and emitters."""
    R = torch.linalg.vector_norm(p, dim=1)
    out = torch.zeros(len(p), dtype=torch.complex128, device="cuda")
    scale = "scale" in case["settings"]
    a = torch.ones(len(e), dtype=torch.float64, device="cuda") if a is None else a.double()
    dn = 1 << 17
    for j in range(0, len(e), dn):
        es, w = e[j:j + dn], a[j:j + dn]
        dp = max(1, (1 << 25) // len(es))
        for i in range(0, len(p), dp):
            th, D = _phases(case, p[i:i + dp], es)
            if scale and " nf" in case["settings"]:
                re, im = (torch.cos(th) / D) @ w, (torch.sin(th) / D) @ w
            else:
                re, im = torch.cos(th) @ w, torch.sin_(th) @ w
            out[i:i + dp] += torch.complex(re, im)
    if scale and " nf" not in case["settings"]:
        out /= R
    if " nf" in case["settings"]:
        ph = K * (p[:, 0] ** 2 + p[:, 1] ** 2) / (R + p[:, 2])
        out *= torch.complex(torch.cos(ph), torch.sin(ph))
    return out


def _gradients(case, e, a, p, field, up):
    """d/d(position, phase, amplitude) of sum(up * |E|^2), the 1/r amplitude held."""
    a1 = torch.ones(len(e), dtype=torch.float64, device="cuda") if a is None else a.double()
    near = " nf" in case["settings"]
    R = torch.linalg.vector_norm(p, dim=1)
    f = field
    if near:
        ph = K * (p[:, 0] ** 2 + p[:, 1] ** 2) / (R + p[:, 2])
        f = field * torch.complex(torch.cos(ph), -torch.sin(ph))
    w = 2 * up.double().reshape(-1) * f.conj()
    gpos, gph, gam = [torch.zeros(s, dtype=torch.float64, device="cuda") for s in ((len(e), 3), (len(e),), (len(e),))]
    dp = max(1, (1 << 25) // len(e))
    for i in range(0, len(p), dp):
        q, ws = p[i:i + dp], w[i:i + dp]
        th, D = _phases(case, q, e)
        c, s = torch.cos(th), torch.sin(th)
        im = -(ws.imag[:, None] * c + ws.real[:, None] * s)  # Re(i w e^{i theta})
        gam += ws.real @ c - ws.imag @ s
        gph += im.sum(0)
        if near:  # d theta / d r = k ((r - p) / D + z)
            v = im / D
            gpos += K * (e[:, :3] * v.sum(0)[:, None] - v.T @ q)
            gpos[:, 2] += K * im.sum(0)
        else:
            Rq = R[i:i + dp, None]
            u = q / Rq
            u[:, 2] = -(q[:, 0] ** 2 + q[:, 1] ** 2) / (Rq[:, 0] * (Rq[:, 0] + q[:, 2]))
            gpos -= K * (im.T @ u)
            if "secondorder" in case["settings"]:
                gpos[:, :2] += (K / Rq * im).sum(0)[:, None] * e[:, :2]
    return gpos * a1[:, None], gph * a1, gam


def _time(case, e, times, p, c, tau):
    """Integral of |E(t)|^2 for emitters that decay with tau from their arrival on."""
    out = torch.empty(len(p), dtype=torch.float64, device="cuda")
    n = len(e)
    for i in range(0, len(p), max(1, (1 << 24) // n)):
        sl = slice(i, i + max(1, (1 << 24) // n))
        th, _ = _phases(case, p[sl], e)
        path = (th - e[:, 3]) / K  # the path difference; minus q.r / k in the far field
        t = path / c + times
        t, order = torch.sort(t, dim=1, stable=True)
        th = torch.gather(th, 1, order)
        x = torch.complex(torch.cos(th), torch.sin(th))
        step = 1
        while step < n:  # inclusive scan of x_i = a_i + exp(-(t_i - t_{i-1}) / tau) x_{i-1}
            decay = torch.exp((t[:, :-step] - t[:, step:]) / tau)
            x = torch.cat([x[:, :step], x[:, step:] + decay * x[:, :-step]], 1)
            step *= 2
        m = x.real ** 2 + x.imag ** 2
        out[sl] = tau / 2 * (m[:, -1] - (m[:, :-1] * torch.expm1(-2 * (t[:, 1:] - t[:, :-1]) / tau)).sum(1))
    return out.reshape(case["n0"], case["n1"])


def _qcorr(case, img):
    """Sum over pixel pairs into bins of the momentum difference; the bins are defined in float32."""
    nr, nc = img.shape
    xc, yc, qmax = nr / 2, nc / 2, max(32, min(1024, case["maxq"], nr, nc))
    zd, maxdqz = _ewald(case)
    zd = torch.from_numpy(zd).cuda()
    f32 = dict(dtype=torch.float32, device="cuda")
    qx = (torch.arange(nr, **f32) - xc)[:, None] * zd
    qy = (torch.arange(nc, **f32) - yc)[None, :] * zd
    sz, sq = 2 * maxdqz, 2 * qmax
    out = torch.zeros(sz * sq * sq, dtype=torch.float64, device="cuda")
    v = img.double()
    cz = torch.tensor(case["z"], **f32)
    oc = torch.arange(1 - qmax, qmax, device="cuda")
    tc = torch.arange(nc, device="cuda")[:, None] + oc  # (column, column offset): neighbours fall in different bins
    inside = (tc >= 0) & (tc < nc)
    tc = tc.clamp(0, nc - 1)
    for dr in range(min(qmax, nr)):
        a, b = slice(0, nr - dr), slice(dr, nr)
        bx = qmax + torch.round(qx[b][:, tc] - qx[a][:, :, None]).long()
        by = qmax + torch.round(qy[b][:, tc] - qy[a][:, :, None]).long()
        bz = maxdqz + torch.round(cz * (zd[a][:, :, None] - zd[b][:, tc])).long()
        ok = inside & (bx >= 0) & (bx < sq) & (by >= 0) & (by < sq) & (bz >= 0) & (bz < sz)
        out.index_add_(0, ((bz * sq + by) * sq + bx)[ok], (v[a][:, :, None] * v[b][:, tc])[ok])
    out = out.reshape(sz, sq, sq)
    mirror = torch.roll(torch.flip(out, (0, 1, 2)), (1, 1, 1), (0, 1, 2))  # entry i holds out[-i mod shape]
    both = out + mirror
    both[:, :, qmax] = out[:, :, qmax]  # bins from the middle on are set from the first half: index qmax has no partner
    return both


def exact(case, seed):
    kind = case["kind"]
    if kind == "photons":
        return None
    x = _inputs(case, seed)
    if kind == "qcorr":
        return _qcorr(case, x["image"]).cpu().numpy()
    p = _pixels(case)
    pairs = len(p) * len(x["emit"])
    if pairs > 1.5e11:
        return None
    shape = (case["n0"], case["n1"])
    if kind == "time":
        return _time(case, x["emit"], x["times"], p, 0.299792458, 1e-3)
    if kind == "shots":
        o = x["offsets"]
        f = torch.stack([_field(case, x["emit"][o[s]:o[s + 1]], x["amp"][o[s]:o[s + 1]] if "amp" in x else None,
                                p).reshape(shape) for s in range(len(o) - 1)])
        return f.real ** 2 + f.imag ** 2 if case["intensity"] else f
    e, a = x["emit"], x.get("amp")
    if kind == "grad":
        e = torch.cat([x["pos"].double(), x["phase"].double()[:, None]], 1)
    f = _field(case, e, a, p)
    if kind == "image":
        f = f.reshape(shape)
        return f.real ** 2 + f.imag ** 2 if case["intensity"] else f
    inten = f.real ** 2 + f.imag ** 2
    if kind == "fit":
        d = inten - x["target"].double().reshape(-1)
        gpos, gph, _ = _gradients(case, e, None, p, f, 2 * d)
        return {"loss": (d * d).sum(), "pos": gpos, "phase": gph}
    gpos, gph, gam = _gradients(case, e, a, p, f, x["up"])
    return {"intensity": inten.reshape(shape), "grads": [gpos, gph] + ([gam] if a is not None else [])}
