"""Gradients of deflector lists by adjoint and per-deflector kernels
(mp_adjoint_kernel, bulk_adjoint_kernel, defl_grad_kernel in csrc/lensim.hip)
at the edges of their pieces: list lengths around a pair and a run, ray counts
around a wave, rays that take several rounds, halos from far inside to far
outside their scale radius."""

import numpy as np
import pytest
import torch

from jaxtronomy_amd import backend
from jaxtronomy_amd import workloads as W
from jaxtronomy_amd.Data.imaging_data import ImageData
from jaxtronomy_amd.Data.psf import PSF
from jaxtronomy_amd.ImSim.image_model import ImageModel
from jaxtronomy_amd.LensModel.lens_model import LensModel
from jaxtronomy_amd.LensModel.lens_model_bulk import LensModelBulk
from jaxtronomy_amd.LightModel.light_model import LightModel

pytestmark = pytest.mark.gpu

UNIQUE = ["EPL", "SHEAR", "TNFW", "CONVERGENCE", "NFW"]
SOURCE = [dict(amp=30.0, R_sersic=0.5, n_sersic=1.3, e1=0.1, e2=-0.05, center_x=0.1, center_y=-0.08)]


def model(num_pix, s, multi_plane, data=None):
    cfg = dict(W.EPL180, numPix=num_pix, deltaPix=3.2 / num_pix, supersampling=s)
    psf = PSF("PIXEL", kernel_point_source=W.moffat_kernel(3, 1.2, 3.0))
    return ImageModel(ImageData(**W.data_kwargs(cfg, data)), psf, LensModelBulk(UNIQUE, multi_plane=multi_plane),
                      LightModel(["SERSIC_ELLIPSE"]), kwargs_numerics={"supersampling_factor": s})


def scene(n_halo, rs, others, seed):
    rng = np.random.default_rng(seed)
    names, kw, z = [], [], []
    if others:  # an EPL and a SHEAR, a sheet, and an NFW in the list
        names += ["EPL", "SHEAR", "CONVERGENCE", "NFW"]
        kw += [dict(theta_E=0.9, gamma=2.05, e1=0.06, e2=-0.04, center_x=0.01, center_y=0.02),
               dict(gamma1=0.02, gamma2=-0.01, ra_0=0.0, dec_0=0.0), dict(kappa=0.03, ra_0=0.0, dec_0=0.0),
               dict(Rs=1.1, alpha_Rs=0.05, center_x=0.3, center_y=-0.2)]
        z += [0.5, 0.5, 0.3, 0.4]
    for i in range(n_halo):
        r = rs * rng.uniform(0.6, 1.6)
        names.append("TNFW")
        kw.append(dict(Rs=r, alpha_Rs=0.15 * min(r, 0.5) / max(1, n_halo) ** 0.5, r_trunc=r * rng.uniform(0.6, 6.0),
                       center_x=rng.uniform(-1, 1), center_y=rng.uniform(-1, 1)))
        z.append(rng.choice([0.3, 0.5, 0.6]))
    return names, kw, z


def packed(im, names, kw, z, multi_plane):
    extra = dict(z_source=1.5, lens_redshift_list=z) if multi_plane else {}
    rs = im.LensModel.prepare_ray_shooting_kwargs(names, kw, **extra)
    return im.pack_bulk(rs, SOURCE)


@pytest.mark.parametrize("multi_plane", [False, True])
@pytest.mark.parametrize("n_halo,rs,num_pix,s,others", [(1, 0.05, 8, 1, False), (2, 3.0, 9, 2, False),
                                                        (65, 0.3, 11, 1, False), (3, 1.0, 12, 2, True),
                                                        (66, 0.02, 23, 1, True)])
def test_list_gradient_vs_differences(n_halo, rs, num_pix, s, others, multi_plane):
    """Every kwarg against central differences of the FP64 logL, which is held to 1e-10 of the oracle: the step h
    leaves a truncation error of h^2 f'''/6 and a rounding error of 1e-16 |logL| / h, so 2e-5 of each kind's scale."""
    names, kw, z = scene(n_halo, rs, others, 7)
    probe = model(num_pix, s, multi_plane)
    params, n, m, keep = packed(probe, names, kw, z, multi_plane)
    clean = probe.image_batch(backend.to_device_f64(params), n, model=m)[0].cpu().numpy()
    im = model(num_pix, s, multi_plane, 1.02 * clean + np.random.default_rng(1).normal(0, 0.02, clean.shape))
    params, n, m, keep = packed(im, names, kw, z, multi_plane)
    pt = backend.to_device_f64(params)
    logl, grad = im.likelihood_and_grad_batch(pt, n, model=m)
    assert torch.allclose(logl, im.likelihood_batch(pt, n, model=m), rtol=1e-12, atol=0.0)
    got = grad[0].cpu().numpy()
    n_prof, want = params.shape[1], np.zeros_like(got)
    moved = [(k, i) for k in range(n_prof) for i in range(8) if got[k, i] != 0.0]
    assert len(moved) >= 3 * (n_prof - 1)
    h = 1e-5
    for at in range(0, len(moved), 128):
        part = moved[at:at + 128]
        batch = np.repeat(params, 2 * len(part), axis=0)
        step = np.array([h * max(abs(params[0, k, i]), 0.05) for k, i in part])
        for b, (k, i) in enumerate(part):
            batch[2 * b, k, i] += step[b]
            batch[2 * b + 1, k, i] -= step[b]
        ll = im.likelihood_batch(backend.to_device_f64(batch), len(batch), model=m).cpu().numpy()
        for b, (k, i) in enumerate(part):
            want[k, i] = (ll[2 * b] - ll[2 * b + 1]) / (2 * step[b])
    scale = np.max(np.abs(got), axis=0)
    assert np.all(np.abs(got - want) <= 2e-5 * np.maximum(scale, 1e-3)), np.max(np.abs(got - want) / (scale + 1e-300))
    del keep


def test_rounds_add_up():
    """A batch whose adjoints take several rounds against the same image alone (one round)."""
    rng = np.random.default_rng(3)
    n = 60
    names, kw, _ = scene(n, 0.2, False, 5)
    z = list(np.sort(rng.uniform(0.1, 1.2, n)))
    im = model(100, 1, True, rng.normal(0.5, 0.1, (100, 100)))
    params, b, m, keep = packed(im, names, kw, z, True)
    l1, g1 = im.likelihood_and_grad_batch(backend.to_device_f64(params), 1, model=m)
    many = backend.to_device_f64(np.repeat(params, 64, axis=0))
    l2, g2 = im.likelihood_and_grad_batch(many, 64, model=m)
    scale = g1.abs().amax(dim=1, keepdim=True).clamp_min(1e-300)
    assert torch.allclose(l2, l1.expand(64), rtol=1e-13, atol=0.0)
    assert float(((g2 - g1) / scale).abs().max()) < 1e-12
    del keep


def test_more_rays_than_an_int_holds():
    """The gradient of a list over more than 2^31 sub-rays, against the same deflector inline, whose kernels go pixel by
    pixel: the sums of a pixel's sub-rays in another order, 2.4e9 terms rounded to 1e-16 each in blocks of at most 1e6."""
    n, s = 4096, 12
    cfg = dict(W.EPL180, numPix=n, deltaPix=3.2 / n, supersampling=s)
    data = np.random.default_rng(0).normal(0.5, 0.1, (n, n))
    halo = dict(Rs=0.6, alpha_Rs=0.4, r_trunc=1.5, center_x=0.013, center_y=0.021)
    grads = []
    for lm in (LensModelBulk(["TNFW"]), LensModel(["TNFW"])):
        im = ImageModel(ImageData(**W.data_kwargs(cfg, data)), PSF("NONE"), lm, LightModel(["SERSIC_ELLIPSE"]),
                        kwargs_numerics={"supersampling_factor": s})
        if isinstance(lm, LensModelBulk):
            params, b, m, keep = im.pack_bulk(lm.prepare_ray_shooting_kwargs(["TNFW"], [halo]), SOURCE)
        else:
            (params, b), m, keep = im.pack([halo], SOURCE), None, None
        grads.append(im.likelihood_and_grad_batch(backend.to_device_f64(params), b, model=m)[1][0].cpu().numpy())
        del im, keep
        torch.cuda.empty_cache()
    assert n * n * s * s > 2**31
    assert np.all(np.abs(grads[0] - grads[1]) <= 1e-9 * np.abs(grads[1]).max(axis=1, keepdims=True))


def test_bound_on_the_plane_runs():
    """The gradient does not depend on the bound that the caller gives on the runs, down to the runs there are; with
    fewer the deflectors' gradients are NaN."""
    names, kw, _ = scene(30, 0.2, False, 5)
    z = [0.3] * 12 + [0.5] * 10 + [0.6] * 8
    im = model(31, 2, True, np.random.default_rng(3).normal(0.5, 0.1, (31, 31)))
    params, n, m, keep = packed(im, names, kw, z, True)
    mp = keep[-1]["struct"]
    assert mp.max_runs == 3

    def grad():
        return im.likelihood_and_grad_batch(backend.to_device_f64(params), n, model=m)[1]

    want = grad()
    for runs in (0, 4, 29, 1 << 20):
        mp.max_runs = runs
        assert torch.equal(grad(), want)
    mp.max_runs = 2
    got = grad()
    assert bool(torch.isnan(got[0, :30]).all()) and torch.equal(got[0, 30:], want[0, 30:])


def test_planes_of_one_redshift_equal_one_plane():
    """More rays than a round's store holds for a run (2^25): several planes at one redshift against the list on one
    plane, whose reduced deflections are the same; 3.4e7 rays' sums in another order, 1e-12 of their sizes."""
    names, kw, _ = scene(3, 0.6, False, 5)
    grads = []
    for multi_plane in (False, True):
        cfg = dict(W.EPL180, numPix=1450, deltaPix=3.2 / 1450, supersampling=4)
        data = np.random.default_rng(0).normal(0.5, 0.1, (1450, 1450))
        im = ImageModel(ImageData(**W.data_kwargs(cfg, data)), PSF("NONE"), LensModelBulk(UNIQUE, multi_plane=multi_plane),
                        LightModel(["SERSIC_ELLIPSE"]), kwargs_numerics={"supersampling_factor": 4})
        params, n, m, keep = packed(im, names, kw, [0.5] * 3, multi_plane)
        grads.append(im.likelihood_and_grad_batch(backend.to_device_f64(params), n, model=m)[1][0].cpu().numpy())
    scale = np.abs(grads[0]).max(axis=1, keepdims=True)
    assert np.all(np.abs(grads[0] - grads[1]) <= 1e-9 * scale)


@pytest.mark.parametrize("n_halo,num_pix", [(3, 40), (40, 61)])
def test_list_gradient_is_the_same_in_any_batch(n_halo, num_pix):
    """The sums' order on one plane follows the image alone."""
    names, kw, _ = scene(n_halo, 0.3, True, 5)
    im = model(num_pix, 1, False, np.random.default_rng(3).normal(0.5, 0.1, (num_pix, num_pix)))
    params, n, m, keep = packed(im, names, kw, None, False)
    alone = im.likelihood_and_grad_batch(backend.to_device_f64(params), n, model=m)
    for b in (2, 37, 300):
        many = im.likelihood_and_grad_batch(backend.to_device_f64(np.repeat(params, b, axis=0)), b, model=m)
        for a, v in zip(alone, many):
            assert torch.equal(v[0], a[0]) and torch.equal(v[-1], a[0])
