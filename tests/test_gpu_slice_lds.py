"""Slice sums whose table just fills a block's LDS (160 KB: 4 B of count and
16 B per term and slice): the largest slice counts that phx_slice_accumulate
takes for each number of terms, one less, where the terms' scales do not fit
either, and one more, which it refuses."""
import numpy as np
import pytest

from tests.test_gpu_slice_blocks import _check

pytestmark = pytest.mark.gpu

LDS = 160 * 1024


@pytest.mark.parametrize("n_terms", range(9))
def test_largest_tables(n_terms):
    from pyheadtail_amd import _phx
    most = LDS // (4 + 16 * n_terms)
    for S in (most, most - 1, most - 24):
        _check(5000, S, n_terms, S % 2 == 0)
    with pytest.raises(_phx.PhxError, match="LDS"):
        _check(5000, most + 1, n_terms, False)


def test_largest_table_of_many_particles():
    _check(300001, LDS // 20, 1, False)


def test_statistics_of_8192_slices():
    """One term per pass: a table of exactly 160 KB."""
    from scipy.constants import e, m_p
    from pyheadtail_amd.particles.particles import Particles
    from pyheadtail_amd.particles.slicing import UniformBinSlicer
    print("\n[case] 8192 slices", flush=True)
    rng = np.random.default_rng(4)
    q = {k: rng.normal(0., 1., 20000) for k in ("x", "xp", "y", "yp", "z", "dp")}
    b = Particles(20000, 1., e, m_p, 6911.5, 27.7, q)
    s = b.get_slices(UniformBinSlicer(8192, n_sigma_z=3), statistics=['mean_x', 'sigma_y'])
    idx = s.slice_index_of_particle.cpu().numpy()
    ok = (idx >= 0) & (idx < 8192)
    n = np.bincount(idx[ok], minlength=8192)
    mean = np.bincount(idx[ok], weights=q['x'][ok], minlength=8192) / np.maximum(n, 1)
    np.testing.assert_allclose(s.mean_x.cpu().numpy(), mean, rtol=0, atol=1e-14)
    my = np.bincount(idx[ok], weights=q['y'][ok], minlength=8192) / np.maximum(n, 1)
    d = q['y'][ok] - my[idx[ok]]
    var = np.bincount(idx[ok], weights=d * d, minlength=8192) / np.maximum(n - 1, 1)
    np.testing.assert_allclose(s.sigma_y.cpu().numpy()[n > 1], np.sqrt(var)[n > 1], rtol=1e-12)
