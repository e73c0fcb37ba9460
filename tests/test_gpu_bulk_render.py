"""Images of bulk deflector lists whose pixels are shared by several waves
(render_bulk_kernel in csrc/lensim.hip) against the oracle, at the list lengths
where the number of waves changes, ragged blocks of 64 pixels, lists of one and
of several types, and with and without lens light."""

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


# of the image's maximum: the library's bars for subhalo images
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-10), ("mixed", 1e-5)])
@pytest.mark.parametrize("n_halo,num_pix,s,nfw,light", [(15, 9, 1, False, False), (16, 9, 3, False, True),
                                                        (17, 31, 2, True, True), (33, 8, 2, False, False),
                                                        (67, 20, 1, True, False), (131, 11, 2, False, True)])
def test_shared_list_image_vs_oracle(n_halo, num_pix, s, nfw, light, precision, tol):
    rng = np.random.default_rng(n_halo)
    cfg = dict(W.EPL180, numPix=num_pix, deltaPix=3.2 / num_pix, supersampling=s)
    kl, ks, kll = W.epl180_draw(7)
    names, kw = ["EPL", "SHEAR"], list(kl)
    for _ in range(n_halo):
        rs = rng.uniform(0.02, 0.4)
        names.append("TNFW")
        kw.append(dict(Rs=rs, alpha_Rs=0.05 * rs, r_trunc=rng.uniform(0.5, 8) * rs, center_x=rng.uniform(-2, 2),
                       center_y=rng.uniform(-2, 2)))
    if nfw:
        names.append("NFW")
        kw.append(dict(Rs=0.9, alpha_Rs=0.1, center_x=0.3, center_y=-0.2))
    ll = ["SERSIC_ELLIPSE"] if light else []
    kernel = W.moffat_kernel(5, 2.0, 3.0)
    im = ImageModel(ImageData(**W.data_kwargs(cfg)),
                    PSF("PIXEL", kernel_point_source=kernel),
                    LensModelBulk(["EPL", "SHEAR", "TNFW", "NFW"], precision=precision), LightModel(["SERSIC_ELLIPSE"]),
                    lens_light_model_class=LightModel(ll), kwargs_numerics={"supersampling_factor": s},
                    precision=precision)
    kwll = [dict(kll[0])] if light else []
    rs = im.LensModel.prepare_ray_shooting_kwargs(names, kw)
    got = im.image(rs, ks, kwll).cpu().numpy()
    want = O.image(W.grid_dict(cfg), names, kw, ["SERSIC_ELLIPSE"], ks, ll, kwll, kernel=kernel)
    assert np.max(np.abs(got - want)) <= tol * np.max(np.abs(want))


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n_halo,nfw", [(17, True), (33, False), (70, False), (140, True)])
def test_same_bits_alone_and_in_a_batch_that_fills_the_chip(n_halo, nfw, precision):
    """2, 4 and 8 classes shared by a block's waves (two images) and in turn in one wave (many)."""
    num_pix, n_img = 40, 260  # 6500 waves of pixels
    rng = np.random.default_rng(n_halo)
    cfg = dict(W.EPL180, numPix=num_pix, deltaPix=0.08, supersampling=1)
    kl, ks, _ = W.epl180_draw(7)
    names, kw = ["EPL", "SHEAR"] + ["TNFW"] * n_halo + ["NFW"] * nfw, list(kl)
    for _ in range(n_halo):
        rs = rng.uniform(0.02, 0.4)
        kw.append(dict(Rs=rs, alpha_Rs=0.05 * rs, r_trunc=4.0 * rs, center_x=rng.uniform(-2, 2),
                       center_y=rng.uniform(-2, 2)))
    if nfw:
        kw.append(dict(Rs=0.9, alpha_Rs=0.1, center_x=0.3, center_y=-0.2))
    data = rng.normal(0.5, 0.1, (num_pix, num_pix))
    im = ImageModel(ImageData(**W.data_kwargs(cfg, data)), PSF("NONE"),
                    LensModelBulk(["EPL", "SHEAR", "TNFW", "NFW"], precision=precision), LightModel(["SERSIC_ELLIPSE"]),
                    precision=precision)
    params, _, m, keep = im.pack_bulk(im.LensModel.prepare_ray_shooting_kwargs(names, kw), ks)
    many = np.repeat(params, n_img, axis=0)
    many[:, 0, 0] *= 1.0 + 1e-3 * np.arange(n_img)
    many = backend.to_device_f64(many)
    two = many[:2].contiguous()
    assert torch.equal(im.image_batch(many, n_img, model=m)[:2], im.image_batch(two, 2, model=m))
    for a, b in zip(im.likelihood_and_grad_batch(many, n_img, model=m), im.likelihood_and_grad_batch(two, 2, model=m)):
        assert torch.equal(a[:2], b)
    del keep
