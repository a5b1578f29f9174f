"""Slice statistics of thin slices.  The covariance of a slice of two or three
macroparticles is singular and its emittance the root of what the sums round
to, so the sums are those of a fixed quantum, 2^(ilogb(bound) - 60) with bound
the product of the factors' max |u| (twice that for a centred factor): every
term to its nearest multiple, ties to even, the whole numbers added, the upper
and the lower 32 bits of the total converted one by one.  Here they are formed
with Python's whole numbers and compared bit for bit, NaN in the same slices."""
import math
from fractions import Fraction

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

COORD = ("x", "xp", "y", "yp", "z", "dp")


def _sum(terms, bound):
    e = 60 - (math.frexp(bound)[1] - 1)
    q = sum(round(Fraction(float(u)) * Fraction(2)**e) for u in terms)
    return math.ldexp(float(q >> 32) * 2.**32 + float(q & 0xffffffff), -e)


def _bunch(n, seed):
    from scipy.constants import e, m_p
    from pyheadtail_amd.particles.particles import Particles
    rng = np.random.default_rng(seed)
    q = {k: rng.normal(0., s, n) for k, s in zip(COORD, (2e-3, 4e-5, 2e-3, 4e-5, 0.23, 1e-3))}
    return Particles(n, 1., e, m_p, 6911.5, 27.7, q), q


@pytest.mark.parametrize("later", [False, True])
@pytest.mark.parametrize("n,S", [(1, 3), (700, 1000), (3000, 333), (5003, 1000)])
def test_thin_slices(n, S, later):
    from scipy.constants import e
    from pyheadtail_amd.particles.slicing import UniformBinSlicer
    print("\n[case] statistics of thin slices: n=%d S=%d later=%s" % (n, S, later), flush=True)
    b, q = _bunch(n, n)
    cuts = dict(z_cuts=(-1., 1.)) if n == 1 else dict(n_sigma_z=3)
    slicer = UniformBinSlicer(S, **cuts)
    if later:
        s = b.get_slices(slicer)
        slicer.add_statistics(s, b, True)
    else:
        s = b.get_slices(slicer, statistics=True)
    idx = s.slice_index_of_particle.cpu().numpy()
    peak = {k: np.abs(q[k]).max() for k in COORD}
    members = [np.flatnonzero(idx == i) for i in range(S)]
    count = np.array([len(m) for m in members])
    mean = {k: np.array([_sum(q[k][m], peak[k]) / len(m) if len(m) else 0. for m in members])
            for k in COORD}
    for k in COORD:
        np.testing.assert_array_equal(getattr(s, "mean_" + k).cpu().numpy(), mean[k], err_msg=k)

    def cov(a, c):
        out = np.zeros(S)
        for i, m in enumerate(members):
            if len(m):
                t = (q[a][m] - mean[a][i]) * (q[c][m] - mean[c][i])
                out[i] = _sum(t, 2 * peak[a] * (2 * peak[c])) / max(1, len(m) - 1)
        return out

    with np.errstate(invalid="ignore", divide="ignore"):
        for k in ("x", "y", "z", "dp"):
            np.testing.assert_array_equal(getattr(s, "sigma_" + k).cpu().numpy(),
                                          np.sqrt(cov(k, k)), err_msg=k)
        d = cov("dp", "dp")
        for name, u, up, disp, f in (("eff_epsn_x", "x", "xp", False, b.betagamma),
                                     ("eff_epsn_y", "y", "yp", False, b.betagamma),
                                     ("epsn_x", "x", "xp", True, b.betagamma),
                                     ("epsn_y", "y", "yp", True, b.betagamma),
                                     ("epsn_z", "z", "dp", False, None)):
            s11, s12, s22 = cov(u, u), cov(u, up), cov(up, up)
            if disp:
                a, c = cov(u, "dp"), cov(up, "dp")
                s11, s12, s22 = (np.where(d != 0., v - w / d, v) for v, w in
                                 ((s11, a * a), (s12, a * c), (s22, c * c)))
            want = np.where(count > 1, np.sqrt(s11 * s22 - s12 * s12), 0.)
            want = want * f if f else 4. * np.pi * want * b.p0 / e
            got = getattr(s, name).cpu().numpy()
            np.testing.assert_array_equal(np.isnan(got), np.isnan(want), err_msg=name)
            np.testing.assert_array_equal(got, want, err_msg=name)
    if n > 1:
        assert np.isnan(got).any() and (got[count == 2] > 0).any()
