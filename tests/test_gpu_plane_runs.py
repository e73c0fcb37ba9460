"""Multi-plane ray shooting by runs of deflectors on one plane (block_trace and
mp_runs_kernel in csrc/lensim.hip) at the lengths where a run is cut, against
the oracle's plane scan."""

import numpy as np
import pytest
import torch

from jaxtronomy_amd import backend
from jaxtronomy_amd import workloads as W
from jaxtronomy_amd.Data.imaging_data import ImageData
from jaxtronomy_amd.Data.psf import PSF
from jaxtronomy_amd.ImSim.image_model import ImageModel
from jaxtronomy_amd.LensModel.lens_model_bulk import LensModelBulk
from jaxtronomy_amd.LightModel.light_model import LightModel
from oracle import lensim_oracle as O

pytestmark = pytest.mark.gpu
FP64_TOL = 1e-10  # of the largest deflection: the library's FP64 bar
UNIQUE = ["TNFW", "CONVERGENCE", "SIE"]


def scene(counts, with_sie, seed):
    """counts[i] TNFW halos on plane i, a sheet on every second plane, and an SIE on the last one when asked for."""
    rng = np.random.default_rng(seed)
    names, kw, z = [], [], []
    for i, n in enumerate(counts):
        for _ in range(n):
            rs = rng.uniform(0.01, 0.4)
            names.append("TNFW")
            kw.append(dict(Rs=rs, alpha_Rs=0.02 * rs, r_trunc=rng.uniform(0.5, 8) * rs, center_x=rng.uniform(-3, 3),
                           center_y=rng.uniform(-3, 3)))
            z.append(0.1 + 0.2 * i)
        if i % 2:
            names.append("CONVERGENCE")
            kw.append(dict(kappa=-0.01, ra_0=0.0, dec_0=0.0))
            z.append(0.1 + 0.2 * i)
    if with_sie:
        names.append("SIE")
        kw.append(dict(theta_E=0.8, e1=0.1, e2=-0.05, center_x=0.02, center_y=-0.01))
        z.append(0.1 + 0.2 * (len(counts) - 1))
    return names, kw, z


@pytest.mark.parametrize("n_ray", [1, 64, 65, 200])
@pytest.mark.parametrize("counts,with_sie", [((1,), False), ((63, 64, 65), False), ((64, 130, 1, 2), True),
                                             ((200,), True)])
def test_runs_vs_oracle(counts, with_sie, n_ray):
    names, kw, z = scene(counts, with_sie, 3)
    rng = np.random.default_rng(n_ray)
    x, y = rng.uniform(-3, 3, n_ray), rng.uniform(-3, 3, n_ray)
    lm = LensModelBulk(UNIQUE, multi_plane=True)
    rs = lm.prepare_ray_shooting_kwargs(names, kw, z_source=2.0, lens_redshift_list=z, num_deflectors=len(names) + 3)
    order = np.argsort(np.array(z))
    n = len(names)
    keep = slice(0, n + 1)
    bx, by = O.multi_plane_ray_shooting(x, y, [names[i] for i in order], [kw[i] for i in order],
                                        rs["T_ij_list"][keep], rs["T_z_list"][keep],
                                        rs["reduced2physical_factor"][keep])
    gx, gy = lm.ray_shooting(x, y, rs)
    scale = max(np.max(np.abs(x - bx)), np.max(np.abs(y - by)))
    err = max(np.max(np.abs(gx.cpu().numpy() - bx)), np.max(np.abs(gy.cpu().numpy() - by)))
    assert err < FP64_TOL * scale


def test_two_models_with_their_own_distances():
    """Plane arrays of their own per batch image (a run ends at other planes in each)."""
    names, kw, _ = scene((78,), False, 5)
    z = [0.1] * 3 + [0.3] * 70 + [0.5] * 5
    z2 = [0.1] * 20 + [0.3] * 53 + [0.5] * 5
    lm = LensModelBulk(UNIQUE, multi_plane=True)
    one = lm.prepare_ray_shooting_kwargs(names, kw, z_source=2.0, lens_redshift_list=z)
    two = lm.prepare_ray_shooting_kwargs(names, kw, z_source=2.0, lens_redshift_list=z2)
    x, y = np.linspace(-2, 2, 70), np.linspace(1, -2, 70)
    bx, by = lm.ray_shooting(x, y, lm.stack_ray_shooting_kwargs([one, two]))
    for i, rs in enumerate((one, two)):
        sx, sy = lm.ray_shooting(x, y, rs)
        assert np.array_equal(bx[i].cpu().numpy(), sx.cpu().numpy())
        assert np.array_equal(by[i].cpu().numpy(), sy.cpu().numpy())


@pytest.mark.parametrize("counts,with_sie,n_img", [((16,), False, 70), ((3, 3, 2), False, 70), ((20, 20), False, 70),
                                                   ((55,) * 20, False, 70), ((3, 2, 1), True, 40), ((30, 40), True, 40),
                                                   ((1, 1, 1, 1), True, 40)])
def test_same_bits_alone_and_in_a_batch_that_fills_the_chip(counts, with_sie, n_img):
    """4, 8 and 16 classes shared by a block's waves (one image) and in turn in one wave (many): images, likelihoods
    and gradients."""
    names, kw, z = scene(counts, with_sie, 9)
    cfg = dict(W.EPL180, numPix=64, deltaPix=0.1, supersampling=1)
    data = np.random.default_rng(0).normal(0.5, 0.1, (64, 64))
    lm = LensModelBulk(UNIQUE, multi_plane=True)
    im = ImageModel(ImageData(**W.data_kwargs(cfg, data)), PSF("NONE"), lm, LightModel(["SERSIC"]))
    rs = lm.prepare_ray_shooting_kwargs(names, kw, z_source=5.0, lens_redshift_list=z)
    params, n, m, keep = im.pack_bulk(rs, [dict(amp=20.0, R_sersic=0.4, n_sersic=1.5, center_x=0.05, center_y=0.03)])
    many = np.repeat(params, n_img, axis=0)
    many[:, 0, 0] *= 1.0 + 1e-3 * np.arange(n_img)
    many = backend.to_device_f64(many)
    two = many[:2].contiguous()
    for call in (im.image_batch, im.likelihood_batch):
        assert torch.equal(call(many, n_img, model=m)[:2], call(two, 2, model=m))
    for a, b in zip(im.likelihood_and_grad_batch(many, n_img, model=m), im.likelihood_and_grad_batch(two, 2, model=m)):
        assert torch.equal(a[:2], b)
    x, y = np.meshgrid(np.linspace(-3, 3, 520), np.linspace(-3, 3, 520))  # 4225 waves of rays
    bx, by = lm.ray_shooting(x, y, rs)
    for i in (0, 519):  # as one image of as many rays, whose order is the same, in another launch
        sx, sy = lm.ray_shooting(np.vstack([x[i:i + 1]] * 2), np.vstack([y[i:i + 1]] * 2), rs)
        scale = float((bx[i] - sx[0]).abs().max()), float((by[i] - sy[0]).abs().max())
        assert max(scale) <= 1e-12
    del keep
