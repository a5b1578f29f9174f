"""A slice of more than 2^24 macroparticles summed by one block, every value
with the same remainder of nearly half a unit of the high limb: the low limbs
alone would pass 2^63, so these engines run four-launch turns, whose histogram
spreads the particles over 256 blocks."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_equal_remainders_of_many_particles():
    from scipy.constants import e, m_p
    from oracle import workloads as W
    from pyheadtail_amd.engine import FusedOneTurnMap
    from pyheadtail_amd.impedances.wakes import CircularResonator, WakeField
    from pyheadtail_amd.particles.particles import Particles
    from pyheadtail_amd.particles.slicing import UniformBinSlicer
    from pyheadtail_amd.trackers.longitudinal_tracking import LinearMap
    n = 2**24 + 2**20
    print("\n[case] one slice of %d macroparticles, one block" % n, flush=True)
    x = (2**25 + 0.499) * 2.**-33      # P = 0 for its bound: units of 2^-33
    q = {k: torch.zeros(n, dtype=torch.float64, device="cuda") for k in ("xp", "y", "yp", "dp")}
    q["x"] = torch.full((n,), x, dtype=torch.float64, device="cuda")
    q["z"] = torch.linspace(-0.1, 0.1, n, dtype=torch.float64, device="cuda")
    b = Particles(n, 1., e, m_p, W.CIRCUMFERENCE, W.GAMMA, q)
    eng = FusedOneTurnMap([LinearMap([W.ALPHA_C], W.CIRCUMFERENCE, 0.017),
                           WakeField(UniformBinSlicer(1, z_cuts=(-1., 1.)),
                                     CircularResonator(1e6, 1e9, 1))],
                          graph_turns=0, pass_grid=1)
    eng.track_turns(b, 4)
    _, counts, mean_x, _ = eng.slice_data
    assert int(counts[0]) == n
    assert abs(float(mean_x[0]) - x) <= 2.**-52 * x
