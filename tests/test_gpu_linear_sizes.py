"""The linear amplitude solve (normal_kernel and lin_solve_kernel, compiled per
number of amplitudes) from one amplitude to the eight it takes, against the
oracle, and two images alone against their batch."""

import numpy as np
import pytest

from jaxtronomy_amd import workloads as W
from jaxtronomy_amd.Data.imaging_data import ImageData
from jaxtronomy_amd.Data.psf import PSF
from jaxtronomy_amd.ImSim.image_linear_solve import ImageLinearFit
from jaxtronomy_amd.LensModel.lens_model import LensModel
from jaxtronomy_amd.LightModel.light_model import LightModel
from oracle import lensim_oracle as O

pytestmark = pytest.mark.gpu


def scene(n_src, n_light, num_pix):
    rng = np.random.default_rng(10 * n_src + n_light)
    kl, ks0, kll0 = W.epl180_draw(4)
    one = lambda amp, r, n, c: dict(amp=amp, R_sersic=r, n_sersic=n, e1=0.05, e2=-0.03, center_x=c[0], center_y=c[1])  # noqa: E731
    ks = [one(20.0 + 5 * i, 0.12 + 0.2 * i, 1.2, rng.uniform(-0.15, 0.15, 2)) for i in range(n_src)]
    kll = [one(10.0 + 3 * i, 0.4 + 0.1 * i, 1.0 + 0.3 * i, rng.uniform(-0.9, 0.9, 2)) for i in range(n_light)]
    cfg = dict(W.EPL180, numPix=num_pix, deltaPix=0.08, supersampling=2)
    return cfg, kl, ks, kll


@pytest.mark.parametrize("n_src,n_light", [(1, 0), (1, 1), (2, 1), (1, 3), (2, 3), (1, 5), (3, 4), (1, 7), (8, 0)])
def test_linear_solve_sizes(n_src, n_light):
    num_pix = 37  # an odd grid of more than one block of 256 pixels, the last one part full
    cfg, kl, ks, kll = scene(n_src, n_light, num_pix)
    kernel = W.moffat_kernel(5, 1.5, 3.0)
    src, light = ["SERSIC_ELLIPSE"] * n_src, ["SERSIC_ELLIPSE"] * n_light
    g = W.grid_dict(cfg)
    clean = O.image(g, ["EPL", "SHEAR"], kl, src, ks, light, kll, kernel=kernel)
    data = W.noisy(clean, cfg["exposure_time"], cfg["background_rms"], np.random.default_rng(2))
    im = ImageLinearFit(ImageData(**W.data_kwargs(cfg, data)), PSF("PIXEL", kernel_point_source=kernel),
                        LensModel(["EPL", "SHEAR"]), LightModel(src), LightModel(light),
                        kwargs_numerics={"supersampling_factor": 2})
    unit = lambda kws: [dict(k, amp=1.0) for k in kws]  # noqa: E731
    logl, amp = im.likelihood_data_given_model(kl, unit(ks), unit(kll), source_marg=True)
    want, want_amp, _, m_inv = O.linear_solve(g, ["EPL", "SHEAR"], kl, src, ks, light, kll, data,
                                              mask=np.ones((num_pix, num_pix)), background_rms=cfg["background_rms"],
                                              exposure_map=cfg["exposure_time"], kernel=kernel, source_marg=True,
                                              linear_prior=None)
    # the normal equations amplify the responses' and sums' rounding (1e-13 of each) by cond(M)
    tol = 1e-13 * np.linalg.cond(np.linalg.inv(m_inv)) * max(1.0, np.max(np.abs(want_amp)))
    assert tol < 1e-2
    assert np.max(np.abs(np.atleast_1d(amp) - want_amp)) <= max(tol, 1e-10 * np.max(np.abs(want_amp)))
    assert abs(float(logl) - want) < 1e-9 * abs(want)
    two = [{k: np.array([v, v * (1.02 if k == "theta_E" else 1.0)]) for k, v in kw.items()} for kw in kl]
    both = im.likelihood_data_given_model(two, unit(ks), unit(kll), source_marg=True)
    assert float(both[0][0]) == float(logl) and np.array_equal(both[1][0], np.atleast_1d(amp))
