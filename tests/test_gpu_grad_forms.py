"""The FP64 gradient's closed forms (epl_dalpha_f64, nie_dalpha_f64,
nfw_dalpha_f64 and sersic_ellipse_grad_f64 in csrc/grad.hpp) where their
branches meet: halos from far inside to far outside their scale radius, cores
from none to large, isothermal and nearly round mass, shallow and steep light."""

import numpy as np
import pytest

from jaxtronomy_amd import backend
from jaxtronomy_amd import workloads as W
from jaxtronomy_amd.Data.imaging_data import ImageData
from jaxtronomy_amd.Data.psf import PSF
from jaxtronomy_amd.ImSim.image_model import ImageModel
from jaxtronomy_amd.LensModel.lens_model import LensModel
from jaxtronomy_amd.LensModel.lens_model_bulk import LensModelBulk
from jaxtronomy_amd.LightModel.light_model import LightModel

pytestmark = pytest.mark.gpu

LENS = {"EPL": dict(theta_E=1.1, gamma=2.05, e1=0.1, e2=-0.07, center_x=0.013, center_y=0.021),
        "SIE": dict(theta_E=1.1, e1=0.1, e2=-0.07, center_x=0.013, center_y=0.021),
        "NIE": dict(theta_E=1.1, e1=0.1, e2=-0.07, s_scale=0.1, center_x=0.013, center_y=0.021),
        "NFW": dict(Rs=1.2, alpha_Rs=0.9, center_x=0.013, center_y=0.021)}
SERSIC = dict(amp=30.0, R_sersic=0.5, n_sersic=1.3, e1=0.1, e2=-0.05, center_x=0.1, center_y=-0.08)


def model(name, num_pix, data=None):
    cfg = dict(W.EPL180, numPix=num_pix, deltaPix=3.2 / num_pix, supersampling=2)
    psf = PSF("PIXEL", kernel_point_source=W.moffat_kernel(3, 1.2, 3.0))
    return ImageModel(ImageData(**W.data_kwargs(cfg, data)), psf, LensModel([name]),
                      LightModel(["SERSIC_ELLIPSE"]), lens_light_model_class=LightModel(["SERSIC_ELLIPSE"]),
                      kwargs_numerics={"supersampling_factor": 2})


@pytest.mark.parametrize("name,lens,light", [
    ("EPL", {}, {}), ("EPL", dict(gamma=2.0), dict(n_sersic=4.0)), ("EPL", dict(e1=0.004, e2=0.003), {}),
    ("SIE", {}, dict(e1=0.0, e2=0.0)), ("NIE", dict(s_scale=1e-3), {}), ("NIE", dict(s_scale=2.0), {}),
    ("NFW", dict(Rs=0.02), {}), ("NFW", dict(Rs=0.3), {}), ("NFW", {}, {}), ("NFW", dict(Rs=30.0), {})])
@pytest.mark.parametrize("num_pix", [5, 23])
def test_gradient_vs_differences(name, lens, light, num_pix):
    """Every kwarg against central differences of the FP64 logL, which is held to 1e-10 of the oracle: the step h
    leaves a truncation error of h^2 f'''/6 and a rounding error of 1e-16 |logL| / h, so 2e-5 of each profile's
    scale (kwargs at 0, where the ellipticity's polar form has no derivative of its own, move by 5e-7)."""
    kw = ([dict(LENS[name], **lens)], [dict(SERSIC, **light)], [dict(SERSIC, amp=12.0, n_sersic=2.2, R_sersic=0.7)])
    probe = model(name, num_pix)
    params, _ = probe.pack(*kw)
    clean = probe.image_batch(backend.to_device_f64(params), 1)[0].cpu().numpy()
    im = model(name, num_pix, 1.02 * clean + np.random.default_rng(1).normal(0, 0.02, clean.shape))
    got = im.likelihood_and_grad_batch(backend.to_device_f64(params), 1)[1][0].cpu().numpy()
    want = np.zeros_like(got)
    n_par = {"EPL": 6, "SIE": 5, "NIE": 6, "NFW": 4}[name]
    at = [(0, i) for i in range(n_par)] + [(k, i) for k in (1, 2) for i in range(7)]
    step = np.array([1e-5 * max(abs(params[0, k, i]), 0.05) for k, i in at])
    batch = np.repeat(params, 2 * len(at), axis=0)
    for n, (k, i) in enumerate(at):
        batch[2 * n, k, i] += step[n]
        batch[2 * n + 1, k, i] -= step[n]
    logl = im.likelihood_batch(backend.to_device_f64(batch), len(batch)).cpu().numpy()
    for n, (k, i) in enumerate(at):
        want[k, i] = (logl[2 * n] - logl[2 * n + 1]) / (2 * step[n])
    for k in range(3):
        scale = np.abs(want[k]).max()
        assert scale > 0.0 and np.all(np.abs(got[k] - want[k]) <= 2e-5 * scale)


DEGENERATE = {"EPL": dict(LENS["EPL"], e1=0.0, e2=0.0), "SIE": dict(LENS["SIE"], e1=0.0, e2=0.0),
              "NIE": dict(LENS["NIE"], e1=0.0, e2=0.0), "NFW": LENS["NFW"],
              "TNFW": dict(Rs=0.0, alpha_Rs=0.5, r_trunc=0.0, center_x=0.1, center_y=0.2)}


@pytest.mark.parametrize("where", ["inline", "bulk", "planes"])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_lens_without_a_source_has_no_gradient(where, precision):
    """No ray carries the lens to the image: every kwarg's gradient is exactly 0, also where a factor of the kwargs
    alone (of a round ellipticity, of a halo of size 0) is infinite or undefined."""
    names = list(DEGENERATE)
    kw = [DEGENERATE[n] for n in names]
    z = [0.3, 0.3, 0.4, 0.5, 0.5]
    cfg = dict(W.EPL180, numPix=9, deltaPix=0.3, supersampling=2)
    lm = (LensModelBulk(names, precision=precision) if where == "bulk" else
          LensModel(names, z_source=1.5, lens_redshift_list=z, multi_plane=True, precision=precision)
          if where == "planes" else LensModel(names, precision=precision))
    data = np.random.default_rng(0).normal(1.0, 0.1, (9, 9))
    im = ImageModel(ImageData(**W.data_kwargs(cfg, data)), PSF("NONE"), lm, LightModel([]),
                    lens_light_model_class=LightModel(["SERSIC_ELLIPSE"]), precision=precision,
                    kwargs_numerics={"supersampling_factor": 2})
    if where == "bulk":
        params, n, m, keep = im.pack_bulk(lm.prepare_ray_shooting_kwargs(names, kw), [], [SERSIC])
    else:
        (params, n), m, keep = im.pack(kw, [], [SERSIC]), None, None
    grad = im.likelihood_and_grad_batch(backend.to_device_f64(params), n, model=m)[1][0].cpu().numpy()
    assert np.all(grad[:5] == 0.0) and np.all(np.isfinite(grad)) and np.any(grad[5] != 0.0)
    del keep


@pytest.mark.parametrize("where", ["inline", "bulk"])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_tnfw_of_negative_radii_vs_differences(where, precision):
    """Rs < 0 with r_trunc < 0 holds X at its floor, where alpha is still a function of Rs through rho0 and tau: alpha =
    a (dx, dy) with one number a, so a kwarg's derivative over that by alpha_Rs is (da / d kwarg) alpha_Rs / a, here from
    a's differences: g at X = 1e-3 cancels to 1e-6 of its terms, so a is good to 1e-9 and steps of 1e-2 leave 1e-4."""
    kw = dict(Rs=-0.7, alpha_Rs=0.1, r_trunc=-1.9, center_x=0.05, center_y=-0.03)
    cfg = dict(W.EPL180, numPix=9, deltaPix=0.3, supersampling=1)
    lm = (LensModelBulk if where == "bulk" else LensModel)(["TNFW"], precision=precision)
    data = np.random.default_rng(0).normal(1.0, 0.1, (9, 9))
    im = ImageModel(ImageData(**W.data_kwargs(cfg, data)), PSF("NONE"), lm, LightModel(["SERSIC_ELLIPSE"]),
                    precision=precision)
    if where == "bulk":
        params, n, m, keep = im.pack_bulk(lm.prepare_ray_shooting_kwargs(["TNFW"], [kw]), [SERSIC])
    else:
        (params, n), m, keep = im.pack([kw], [SERSIC]), None, None
    g = im.likelihood_and_grad_batch(backend.to_device_f64(params), n, model=m)[1][0].cpu().numpy()[0]

    def a(rs, rt):  # tnfw.py:226-248 with X = 0.001, up to a constant
        x, tau = 1e-3, rt / rs
        w, t2 = np.sqrt(tau * tau + x * x), tau * tau
        f = np.arctanh(np.sqrt(1 - x * x)) / np.sqrt(1 - x * x)
        return t2 / (t2 + 1)**2 * ((t2 - 1 + 2 * x * x) * f + tau * np.pi + (t2 - 1) * np.log(tau)
                                   + w * (-np.pi + np.log(x / (tau + w)) * (t2 - 1) / tau)) / rs

    h = 1e-2
    by_rs = (a(kw["Rs"] + h, kw["r_trunc"]) - a(kw["Rs"] - h, kw["r_trunc"])) / (2 * h) / a(kw["Rs"], kw["r_trunc"])
    by_rt = (a(kw["Rs"], kw["r_trunc"] + h) - a(kw["Rs"], kw["r_trunc"] - h)) / (2 * h) / a(kw["Rs"], kw["r_trunc"])
    assert g[1] != 0.0
    assert abs(g[0] / (g[1] * kw["alpha_Rs"]) - by_rs) <= 1e-3 * abs(by_rs)
    assert abs(g[2] / (g[1] * kw["alpha_Rs"]) - by_rt) <= 1e-3 * abs(by_rt) + 1e-6
