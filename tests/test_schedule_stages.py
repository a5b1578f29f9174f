"""Turn table of maps with space-charge kicks, whose turns store a program
per stage side by side: each entry is the first of its turn's programs, also
after the turn that leaves the host scalars unchanged (rings whose RF kick
moves p0 in the first turns, or in every turn)."""
import numpy as np
import pytest

from oracle import workloads as W


class _Scalars(object):
    pass


def _beam(gamma):
    b = _Scalars()
    b.mass, b.charge, b.circumference = W.m_p, W.e, W.CIRCUMFERENCE
    b.macroparticlenumber, b.particlenumber_per_mp = 100, 1e9
    b._gamma = gamma
    b._beta = np.sqrt(1 - gamma**-2)
    b._betagamma = np.sqrt(gamma**2 - 1)
    b._p0 = b._betagamma * W.m_p * W.c
    return b


def _ring(gamma, p_increment, n_sc):
    from pyheadtail_amd.particles.slicing import UniformBinSlicer
    from pyheadtail_amd.spacecharge.spacecharge import TransverseGaussianSpaceCharge
    from pyheadtail_amd.trackers.longitudinal_tracking import RFSystems
    from pyheadtail_amd.trackers.transverse_tracking import TransverseMap
    C = W.CIRCUMFERENCE
    n = max(1, n_sc)
    s = np.arange(n + 1) * C / n
    one = np.ones(n + 1)
    segments = TransverseMap(s, 0 * s, W.BETA_X * one, 0 * s, 0 * s, W.BETA_Y * one, 0 * s,
                             W.Q_X, W.Q_Y)
    rf = RFSystems(C, [W.H_RF], [W.V_RF], [0.], [W.ALPHA_C], gamma, p_increment=p_increment,
                   charge=W.e, mass=W.m_p)
    els = [rf]
    for i in range(n):
        els.append(segments[i])
        if i < n_sc:
            els.append(TransverseGaussianSpaceCharge(UniformBinSlicer(20, n_sigma_z=3), C / n))
    return els


@pytest.mark.parametrize("n_sc", [0, 1, 2])
@pytest.mark.parametrize("p_increment", [0., 1e-24])
def test_table_points_at_each_turns_first_program(n_sc, p_increment):
    from pyheadtail_amd.engine import FusedOneTurnMap
    from pyheadtail_amd.particles.particles import ScalarState
    moved = 0
    for gamma in (27.7, 27.728564, 11.3, 100.1, 251.7):
        eng = FusedOneTurnMap(_ring(gamma, p_increment, n_sc))
        progs, table = eng._schedule(_beam(gamma), 30)
        st = ScalarState(_beam(gamma))
        n_st = n_sc + 1
        for t in range(30):
            want = b"".join(bytes(memoryview(q).cast("B")) for q in eng._program(st))
            assert table[t] % n_st == 0
            assert progs[table[t] // n_st] == want, (gamma, t)
        moved += len(progs) > 1
    assert moved > 0


@pytest.mark.gpu
def test_rf_ring_with_space_charge_vs_elements():
    """Seven turns, the program settling in the third: the fused
    stages against the element loop, which shares their arithmetic up to the
    last bits of the slice deviations (bound of the LinearMap ring's test)."""
    print("\n[case] RF ring with fused space charge vs element by element", flush=True)
    import torch
    from pyheadtail_amd import _phx
    from pyheadtail_amd.engine import FusedOneTurnMap
    from pyheadtail_amd.particles.particles import Particles
    from tests.machines import COORDS, clone_bunch, coord_err, to_numpy
    gamma = 11.3            # three programs, the last from the third turn on
    ob = W.nonlinear_bunch(20000, seed=9)
    b = Particles(20000, ob.particlenumber_per_mp, W.e, W.m_p, W.CIRCUMFERENCE, gamma,
                  {k: getattr(ob, k) for k in COORDS})
    b2 = clone_bunch(b)
    ring = _ring(gamma, 0., 2)
    eng = FusedOneTurnMap(ring, graph_turns=4, pass_grid=_phx.STANDALONE_GRID)
    eng.track_turns(b, 7)
    assert len(set(eng._bufs['host_table'][:7])) > 1
    for _ in range(7):
        for el in ring:
            el.track(b2)
    torch.cuda.synchronize()
    ref = type("", (), to_numpy(b2))
    assert coord_err(to_numpy(b), ref) < 1e-12
