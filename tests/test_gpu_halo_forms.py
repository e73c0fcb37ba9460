"""The FP64 TNFW deflection (tnfw_core in csrc/profiles.hpp) on both sides of
each line between its series, against 40-digit arithmetic."""

import mpmath as mp
import numpy as np
import pytest

from jaxtronomy_amd.LensModel.lens_model import LensModel

pytestmark = pytest.mark.gpu


def tnfw_terms(x, tau):
    """The terms of the reference's g (LensModel/Profiles/tnfw.py:329-349) in 40 digits, times its prefactor."""
    with mp.workdps(40):
        x, tau = mp.mpf(float(x)), mp.mpf(float(tau))
        u, t2 = x * x, tau * tau
        s = mp.sqrt(abs(1 - u))
        f = mp.mpf(1) if u == 1 else (mp.atanh(s) if u < 1 else mp.atan(s)) / s
        w = mp.sqrt(t2 + u)
        pre = t2 / (t2 + 1) ** 2
        return [pre * t for t in ((t2 + 2 * u - 1) * f, tau * mp.pi, (t2 - 1) * mp.log(tau), -mp.pi * w,
                                  w * mp.log(x / (tau + w)) * (t2 - 1) / tau)]


@pytest.mark.parametrize("tau", [0.3, 1.0, 1.5, 5.0, 30.0, 500.0])
def test_tnfw_fp64_at_the_lines_between_its_series(tau):
    # the lines: X = 1/2 (P), 2 (G), max(4, 4 tau) (both far series), 2 tau (asinh), and the exact X = 1
    lines = [0.5, 1.0, 2.0, 2.0 * tau, 4.0, 4.0 * tau]
    x = np.array(sorted(v * k for v in lines for k in (0.9, 1 - 1e-9, 1.0, 1 + 1e-9, 1.1) if v * k >= 0.5) +
                 [50.0 * max(1.0, tau), 3e4])
    bx, _ = LensModel(["TNFW"]).ray_shooting(x, np.zeros_like(x), [dict(Rs=1.0, alpha_Rs=1.0, r_trunc=tau,
                                                                       center_x=0.0, center_y=0.0)])
    got = x - bx.cpu().numpy()
    for xi, gi in zip(x, got):
        terms = tnfw_terms(xi, tau)
        with mp.workdps(40):
            scale = 1 / (mp.mpf(float(xi)) * (1 + mp.log(mp.mpf(1) / 2)))
            want = sum(terms) * scale
            # 16 roundings of the sum's terms (as the reference adds them), and that of beta = x - alpha
            tol = float(16 * mp.mpf(2) ** -53 * sum(abs(t) for t in terms) * scale) + 2.0 ** -52 * xi
            assert abs(float(mp.mpf(float(gi)) - want)) <= tol, (tau, xi)
