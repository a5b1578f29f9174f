"""Calls whose turns do not all run the same program (accelerating rings: one
per turn; rings whose p0 settles after some turns): the launch sequences they
take, counted at the library's entry points, and their results, which are
those of single-turn calls (four launches a turn, no graph) bit for bit."""
import numpy as np
import pytest

from oracle import workloads as W

pytestmark = pytest.mark.gpu


def _map(gamma, p_increment):
    from pyheadtail_amd.impedances.wakes import CircularResonator, WakeField
    from pyheadtail_amd.particles.slicing import UniformBinSlicer
    from pyheadtail_amd.trackers.longitudinal_tracking import RFSystems
    from tests.machines import smooth_transverse
    rf = RFSystems(W.CIRCUMFERENCE, [W.H_RF], [W.V_RF], [0.], [W.ALPHA_C], gamma,
                   p_increment=p_increment, charge=W.e, mass=W.m_p)
    return [rf, smooth_transverse(5.)[0],
            WakeField(UniformBinSlicer(50, n_sigma_z=3), CircularResonator(1e6, 1e9, 1))]


def _bunch(gamma, n, seed=3):
    from pyheadtail_amd.particles.particles import Particles
    from tests.machines import COORDS
    ob = W.nonlinear_bunch(n, seed=seed)
    return Particles(n, ob.particlenumber_per_mp, W.e, W.m_p, W.CIRCUMFERENCE, gamma,
                     {k: getattr(ob, k) for k in COORDS})


def _calls(monkeypatch):
    """[(entry point, its count of turns, the engine record's ahead)] from here on."""
    import ctypes
    from pyheadtail_amd import _phx
    seen, call = [], _phx.call

    def counting(fn, *args):
        name = getattr(fn, "__name__", "")
        if name in ("phx_engine_turns", "phx_graph_capture"):
            seen.append((name, args[1], ctypes.cast(args[0], ctypes.POINTER(
                _phx.Engine)).contents.ahead))
        elif name == "phx_graph_launch":
            seen.append((name, None, None))
        return call(fn, *args)
    monkeypatch.setattr(_phx, "call", counting)
    return seen


# gamma, p_increment, turns of the call: launches expected with graphs of 4
ROUTES = [
    (27.728564, 1e-24, 14, [("phx_graph_capture", 4, 0)] + [("phx_graph_launch", None, None)] * 3 +
     [("phx_engine_turns", 2, 0)]),
    (11.3, 0., 11, [("phx_engine_turns", 2, 0), ("phx_graph_capture", 4, 1)] +
     [("phx_graph_launch", None, None)] * 2 + [("phx_engine_turns", 1, 1)]),
    (50.3, 0., 13, [("phx_graph_capture", 4, 0), ("phx_graph_launch", None, None),
                    ("phx_engine_turns", 1, 0), ("phx_graph_capture", 4, 1)] +
     [("phx_graph_launch", None, None)] * 2),
    (50.3, 0., 8, [("phx_graph_capture", 4, 0)] + [("phx_graph_launch", None, None)] * 2),
    (27.728564, 0., 3, [("phx_engine_turns", 3, 0)]),
]


@pytest.mark.parametrize("gamma,p_increment,turns,expected", ROUTES)
def test_launch_sequences_and_results(gamma, p_increment, turns, expected, monkeypatch):
    print("\n[case] gamma %g, p_increment %g, %d turns" % (gamma, p_increment, turns), flush=True)
    from pyheadtail_amd.engine import FusedOneTurnMap
    from tests.machines import COORDS, to_numpy
    one = _bunch(gamma, 20011)
    eng = FusedOneTurnMap(_map(gamma, p_increment), pass_grid=20)
    for _ in range(turns):
        eng.track_turns(one, 1, use_graph=False)
    many = _bunch(gamma, 20011)
    eng = FusedOneTurnMap(_map(gamma, p_increment), graph_turns=4, pass_grid=20)
    seen = _calls(monkeypatch)
    eng.track_turns(many, turns)
    assert seen == expected
    one, many = to_numpy(one), to_numpy(many)
    for k in COORDS:
        np.testing.assert_array_equal(one[k], many[k], err_msg=k)
