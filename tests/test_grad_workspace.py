"""lensim_grad_workspace_size of multi-plane lists and lensim_multiplane.max_runs
(host code alone: nothing is launched)."""

import ctypes

import numpy as np
import pytest

from jaxtronomy_amd import backend, profiles


def grad_bytes(n_defl, runs, n_img, num_pix, precision=0):
    m = backend.make_model([], [profiles.LIGHT_PROFILES["SERSIC_ELLIPSE"][0]], [],
                           bulk=(n_defl, profiles.LENS_PROFILES["TNFW"][0], None))
    mp = backend.LensimMultiplane()
    mp.n_planes, mp.max_runs = n_defl + 1, runs
    mp.d_order = mp.d_T_ij = mp.d_T_z = mp.d_r2p = 4096  # not read
    m.multiplane = ctypes.addressof(mp)
    g = backend.LensimGrid()
    g.nx = g.ny = num_pix
    g.supersampling = 1
    g.pix2angle[0] = g.pix2angle[3] = 0.1
    psf = backend.LensimPsf()
    return backend.lib().lensim_grad_workspace_size(ctypes.byref(m), ctypes.byref(g), ctypes.byref(psf), n_img, precision)


@pytest.mark.parametrize("n_img,num_pix,runs,most", [(1, 100, 130, 100e6), (1, 100, 0, 1.2e9), (64, 100, 130, 2.0e9),
                                                     (64, 100, 0, 2.0e9), (16, 400, 130, 2.0e9), (64, 400, 0, 5e9)])
def test_workspace_of_a_line_of_sight(n_img, num_pix, runs, most):
    """5256 deflectors: the adjoints' store is at most 1 GiB and as large as the runs need; the rest is proportional to
    the images (records, one partial sum per profile and block of pixels, a few per deflector)."""
    assert 0 < grad_bytes(5256, runs, n_img, num_pix) < most


def test_a_bound_of_no_use_counts_a_run_per_deflector():
    for runs in (-1, 5256, 1 << 30):
        assert grad_bytes(5256, runs, 1, 100) == grad_bytes(5256, 0, 1, 100)


def test_plane_runs():
    """A redshift with m deflectors makes ceil(m / 64) runs; the source's plane is none."""
    def arrays(counts):
        t_ij = np.concatenate([np.eye(1, c)[0] * 10.0 for c in counts] + [[5.0]])
        t_z = np.cumsum(t_ij)
        return t_ij, t_z, np.concatenate([np.full(c, 1.0 + i) for i, c in enumerate(counts)] + [[0.0]])

    assert backend.plane_runs(*arrays([1])) == 1
    assert backend.plane_runs(*arrays([1, 1, 1])) == 3
    assert backend.plane_runs(*arrays([64, 65, 128, 2])) == 1 + 2 + 2 + 1
    one, two = arrays([3, 3]), arrays([1, 1, 4])
    assert backend.plane_runs(*[np.stack(v) for v in zip(one, two)]) == 3
    assert backend.plane_runs([1.0], [1.0], [0.0]) == 0
    t_ij, t_z, r2p = arrays([4])
    r2p[2] = 9.0  # another factor, though at the same position
    assert backend.plane_runs(t_ij, t_z, r2p) == 3
