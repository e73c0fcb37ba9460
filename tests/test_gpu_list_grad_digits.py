"""Gradients of deflector lists, every kwarg of every deflector against float64
complex-step derivatives of the model, at the list lengths and ray counts
where the kernels' pieces end (a pair, a run, a wave, a split of the rays)."""

import numpy as np
import pytest

from jaxtronomy_amd import backend
from jaxtronomy_amd.Data.imaging_data import ImageData
from jaxtronomy_amd.Data.psf import PSF
from jaxtronomy_amd.ImSim.image_model import ImageModel
from jaxtronomy_amd.LensModel.lens_model_bulk import LensModelBulk
from jaxtronomy_amd.LightModel.light_model import LightModel

pytestmark = pytest.mark.gpu

SIGMA = 0.05
NAMES = {"SIE": ["theta_E", "e1", "e2", "center_x", "center_y"], "NFW": ["Rs", "alpha_Rs", "center_x", "center_y"],
         "TNFW": ["Rs", "alpha_Rs", "r_trunc", "center_x", "center_y"], "SHEAR": ["gamma1", "gamma2", "ra_0", "dec_0"],
         "CONVERGENCE": ["kappa", "ra_0", "dec_0"]}
UNIQUE = list(NAMES)
SOURCE = dict(amp=30.0, R_sersic=0.5, n_sersic=1.3, e1=0.1, e2=-0.05, center_x=0.1, center_y=-0.08)


def alpha(t, p, x, y):
    if t == "SHEAR":
        dx, dy = x - p[2], y - p[3]
        return p[0] * dx + p[1] * dy, p[1] * dx - p[0] * dy
    if t == "CONVERGENCE":
        return p[0] * (x - p[1]), p[0] * (y - p[2])
    dx, dy = x - p[-2], y - p[-1]
    if t == "SIE":
        c = np.sqrt(p[1] * p[1] + p[2] * p[2])
        q, phi = (1 - c) / (1 + c), np.angle(p[1].real + 1j * p[2].real) / 2
        # cos and sin of the orientation by half angles, analytic in e1, e2
        cs = np.sqrt((1 + p[1] / c) / 2) * np.sign(np.cos(phi))
        sn = p[2] / c / (2 * cs)
        xr, yr = dx * cs + dy * sn, dy * cs - dx * sn
        core = 1e-10 / np.sqrt(q)
        psi, sq = np.sqrt(q * q * (core * core + xr * xr) + yr * yr), np.sqrt(1 - q * q)
        b = p[0] * np.sqrt(q) / sq
        fx, fy = b * np.arctan(sq * xr / (psi + core)), b * np.arctanh(sq * yr / (psi + q * q * core))
        return fx * cs - fy * sn, fx * sn + fy * cs
    u = (dx * dx + dy * dy) / (p[0] * p[0])
    s = np.sqrt(np.where(u.real < 1, 1 - u, u - 1))
    f = np.where(u.real < 1, np.arctanh(np.where(u.real < 1, s, 0.5)), np.arctan(s)) / s
    xx = np.sqrt(u)
    if t == "NFW":
        g = np.log(xx / 2) + f
    else:
        tau = p[2] / p[0]
        t2, w = tau * tau, np.sqrt(tau * tau + u)
        g = t2 / (t2 + 1) ** 2 * ((t2 + 2 * u - 1) * f + tau * np.pi + (t2 - 1) * np.log(tau)
                                  + w * (-np.pi + np.log(xx / (tau + w)) * (t2 - 1) / tau))
    a = p[1] / (p[0] * (1 + np.log(0.5))) * g / u
    return a * dx, a * dy


def flux(p, x, y):
    dx, dy = x - p[5], y - p[6]
    r = np.sqrt((((1 - p[3]) * dx - p[4] * dy) ** 2 + ((1 + p[3]) * dy - p[4] * dx) ** 2) / (1 - p[3]**2 - p[4]**2))
    return p[0] * np.exp(-(1.9992 * p[2] - 0.3271) * (np.exp(np.log(r / p[1]) / p[2]) - 1))


def image(names, ps, src, x, y, planes):
    if planes is None:
        a = [alpha(t, p, x, y) for t, p in zip(names, ps)]
        return flux(src, x - sum(v[0] for v in a), y - sum(v[1] for v in a))
    tij, tz, r2p = planes
    px = py = 0.0
    ax, ay = x, y
    for i, (t, p) in enumerate(zip(names, ps)):
        px, py = px + ax * tij[i], py + ay * tij[i]
        dx, dy = alpha(t, p, px / tz[i], py / tz[i])
        ax, ay = ax - r2p[i] * dx, ay - r2p[i] * dy
    return flux(src, (px + ax * tij[-1]) / tz[-1], (py + ay * tij[-1]) / tz[-1])


def scene(n_halo, rs, others, seed):
    rng = np.random.default_rng(seed)
    names, kw, z = [], [], []
    if others:
        names += ["SIE", "SHEAR", "CONVERGENCE", "NFW"]
        kw += [dict(theta_E=0.9, e1=0.06, e2=-0.04, center_x=0.01, center_y=0.02),
               dict(gamma1=0.02, gamma2=-0.01, ra_0=0.05, dec_0=0.1), dict(kappa=0.03, ra_0=0.02, dec_0=-0.1),
               dict(Rs=1.1, alpha_Rs=0.05, center_x=0.3, center_y=-0.2)]
        z += [0.5, 0.5, 0.3, 0.4]
    for _ in range(n_halo):
        r = rs * rng.uniform(0.6, 1.6)
        names.append("TNFW")
        kw.append(dict(Rs=r, alpha_Rs=0.15 * min(r, 0.5) / max(1, n_halo) ** 0.5, r_trunc=r * rng.uniform(0.6, 6.0),
                       center_x=rng.uniform(-1, 1), center_y=rng.uniform(-1, 1)))
        z.append(rng.choice([0.3, 0.5, 0.6]))
    order = np.argsort(z, kind="stable")
    return [names[i] for i in order], [kw[i] for i in order], [z[i] for i in order]


def build(n, multi_plane, data):
    half, pixel = 1.6 * (n - 1) / n, 3.2 / n
    obs = ImageData(data, noise_map=np.full((n, n), SIGMA), ra_at_xy_0=-half, dec_at_xy_0=-half,
                    transform_pix2angle=pixel * np.eye(2))
    g = pixel * np.arange(n) - half
    return (ImageModel(obs, PSF("NONE"), LensModelBulk(UNIQUE, multi_plane=multi_plane), LightModel(["SERSIC_ELLIPSE"])),
            np.tile(g, n), np.repeat(g, n), pixel**2)


@pytest.mark.parametrize("multi_plane", [False, True])
@pytest.mark.parametrize("n_halo,rs,n,others", [(1, 0.3, 8, False), (2, 1.0, 9, False), (65, 0.3, 11, False),
                                                (3, 1.0, 12, True), (66, 0.1, 23, True), (130, 0.2, 33, True)])
def test_every_kwarg_of_a_list(n_halo, rs, n, others, multi_plane):
    """The kernel's and the reference's halo terms round to 16 2^-53 and cancel to X^2 of themselves, X = 0.02 or more:
    4e-12 of alpha, times the source's second derivatives over its first, below 1e2 here: 1e-9 of the sum over the
    rays of the contributions' absolute values."""
    names, kw, z = scene(n_halo, rs, others, 11)
    extra = dict(z_source=1.5, lens_redshift_list=z) if multi_plane else {}

    def packed(im):
        r = im.LensModel.prepare_ray_shooting_kwargs(names, kw, **extra)
        return (r,) + im.pack_bulk(r, [SOURCE])

    im, x, y, area = build(n, multi_plane, np.zeros((n, n)))
    r, params, _, m, keep = packed(im)
    clean = im.image_batch(backend.to_device_f64(params), 1, model=m)[0].cpu().numpy()
    data = 1.02 * clean + np.random.default_rng(1).normal(0, 0.05, clean.shape)
    im = build(n, multi_plane, data)[0]
    r, params, _, m, keep = packed(im)
    grad = im.likelihood_and_grad_batch(backend.to_device_f64(params), 1, model=m)[1][0].cpu().numpy()
    planes = (r["T_ij_list"], r["T_z_list"], r["reduced2physical_factor"]) if multi_plane else None
    cplx = lambda t, k: np.array([k[v] for v in t], dtype=complex)  # noqa: E731
    ps, src = [cplx(NAMES[t], k) for t, k in zip(names, kw)], cplx(list(SOURCE), SOURCE)
    model = area * image(names, ps, src, x, y, planes).real
    assert np.max(np.abs(model - clean.ravel())) <= 1e-10 * np.max(np.abs(model))
    w = -(model - data.ravel()) / SIGMA**2
    for d, p in enumerate(ps + [src]):
        row = im.LensModel._packed[d] if d < len(ps) else len(ps)
        for i in range(len(p)):
            p[i] += 1e-30j
            v = w * area * image(names, ps, src, x, y, planes).imag / 1e-30
            p[i] -= 1e-30j
            assert abs(grad[row, i] - v.sum()) <= 1e-9 * np.abs(v).sum(), (d, i, grad[row, i], v.sum())
    del keep
