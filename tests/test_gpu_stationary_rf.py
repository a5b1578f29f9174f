"""The stationary RF pass where the kick changes p0: with p_increment = 0 the
round trip p0 -> gamma -> p0 still moves p0's last bit in the first turns of
about half of all rings (three programs for gamma = 11.3, six for 50.3), and
dp is scaled by p0_before / p0_after.  The pass compiled for stationary RF,
the general one, the one that records statistics and a batch's give the same
bits."""
import numpy as np
import pytest

from oracle import workloads as W

pytestmark = pytest.mark.gpu


def _bunch(gamma, n):
    from pyheadtail_amd.particles.particles import Particles
    from tests.machines import COORDS
    ob = W.nonlinear_bunch(n, seed=21)
    return Particles(n, ob.particlenumber_per_mp, W.e, W.m_p, W.CIRCUMFERENCE, gamma,
                     {k: getattr(ob, k) for k in COORDS})


def _map(gamma):
    from pyheadtail_amd.impedances.wakes import CircularResonator, WakeField
    from pyheadtail_amd.particles.slicing import UniformBinSlicer
    from pyheadtail_amd.trackers.longitudinal_tracking import RFSystems
    from tests.machines import smooth_transverse
    rf = RFSystems(W.CIRCUMFERENCE, [W.H_RF], [W.V_RF], [0.], [W.ALPHA_C], gamma, p_increment=0.,
                   charge=W.e, mass=W.m_p)
    return [rf, smooth_transverse(5., 1e-10 * W.P0, -5e-11 * W.P0)[0],
            WakeField(UniformBinSlicer(50, n_sigma_z=3), CircularResonator(1e6, 1e9, 1))]


@pytest.mark.parametrize("gamma", [11.3, 50.3])
@pytest.mark.parametrize("turns", [[1], [2, 9]])
def test_stationary_pass_keeps_the_momentum_ratio(gamma, turns):
    print("\n[case] stationary RF, gamma %g, turns %r" % (gamma, turns), flush=True)
    from pyheadtail_amd import _phx
    from pyheadtail_amd.batch import BatchedScan
    from pyheadtail_amd.engine import FusedOneTurnMap
    from tests.machines import COORDS, to_numpy
    n, out = 30001, {}
    for name, kw in (("stationary", {}), ("general", dict(specialise=False)),
                     ("statistics", dict(record_stats=True))):
        b = _bunch(gamma, n)
        eng = FusedOneTurnMap(_map(gamma), graph_turns=4, pass_grid=40, **kw)
        for k in turns:
            eng.track_turns(b, k)
            if name == "stationary":
                assert eng._shape[0] & _phx.SHAPE_STATIONARY
        out[name] = to_numpy(b)
    jobs = [(_map(gamma), _bunch(gamma, n)), (_map(gamma), _bunch(gamma, 5000))]
    scan = BatchedScan(jobs, graph_turns=4, pass_grid=40)
    for k in turns:
        scan.track_turns(k)
    out["batch"] = to_numpy(scan.bunches[0])
    for name in ("general", "statistics", "batch"):
        for k in COORDS:
            np.testing.assert_array_equal(out["stationary"][k], out[name][k],
                                          err_msg="%s %s" % (name, k))
