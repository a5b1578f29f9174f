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


def _batch_calls(monkeypatch):
    """[(entry point, ahead of each engine or count of turns)] from here on."""
    from pyheadtail_amd import _phx
    seen, call = [], _phx.call

    def counting(fn, *args):
        name = getattr(fn, "__name__", "")
        if name == "phx_batch_create":
            seen.append((name, [args[0][i].ahead for i in range(args[1])]))
        elif name in ("phx_batch_capture", "phx_batch_turns"):
            seen.append((name, args[1]))
        return call(fn, *args)
    monkeypatch.setattr(_phx, "call", counting)
    return seen


def _alone(jobs, turns):
    from pyheadtail_amd.engine import FusedOneTurnMap
    from tests.machines import to_numpy
    out = []
    for m, b in jobs:
        eng = FusedOneTurnMap(m, pass_grid=20, specialise=True)
        for k in turns:
            eng.track_turns(b, k, use_graph=False)
        out.append(to_numpy(b))
    return out


def _check_batch(make, turns, monkeypatch):
    """The jobs in one scan and each alone, bit for bit; the scan's calls."""
    from pyheadtail_amd.batch import BatchedScan
    from tests.machines import COORDS, to_numpy
    want = _alone(make(), turns)
    scan = BatchedScan(make(), graph_turns=4, pass_grid=20)
    seen = _batch_calls(monkeypatch)
    for k in turns:
        scan.track_turns(k)
    for b, w in zip(scan.bunches, want):
        for k, v in to_numpy(b).items():
            if k in COORDS:
                np.testing.assert_array_equal(v, w[k], err_msg=k)
    return seen


def test_scan_with_settling_programs(monkeypatch):
    """Jobs whose programs settle after 0, 2 and 5 turns: five turns of four
    launches for all of them, then three-launch turns, in one batch each."""
    print("\n[case] scan of rings that settle at different turns", flush=True)

    def make():
        return [(_map(g, 0.), _bunch(g, n, n)) for g, n in ((27.728564, 8000), (11.3, 20011),
                                                            (50.3, 1025))]
    seen = _check_batch(make, [14, 9], monkeypatch)
    assert seen == [("phx_batch_create", [0, 0, 0]), ("phx_batch_capture", 4), ("phx_batch_turns", 1),
                    ("phx_batch_create", [1, 1, 1]), ("phx_batch_capture", 4), ("phx_batch_turns", 1),
                    ("phx_batch_turns", 1)]


def test_accelerating_scan(monkeypatch):
    print("\n[case] scan of accelerating rings", flush=True)

    def make():
        return [(_map(g, 1e-24), _bunch(g, n, n)) for g, n in ((27.728564, 8000), (11.3, 20011))]
    seen = _check_batch(make, [10], monkeypatch)
    assert seen == [("phx_batch_create", [0, 0]), ("phx_batch_capture", 4), ("phx_batch_turns", 2)]


@pytest.mark.parametrize("least,created", [(None, [[0, 0]]), (1, [[1], [0]])])
def test_scan_with_and_without_kicks_on_dp(least, created, monkeypatch):
    print("\n[case] scan with and without kicks on dp, least %r" % least, flush=True)
    from pyheadtail_amd import batch
    from pyheadtail_amd.impedances.wakes import Resonator, WakeField
    from pyheadtail_amd.particles.slicing import UniformBinSlicer
    if least is not None:
        monkeypatch.setattr(batch, "MIXED_MIN", least)

    def make():
        jobs = [(_map(27.728564, 0.), _bunch(27.728564, n, n)) for n in (8000, 20011)]
        jobs[1][0][2] = WakeField(UniformBinSlicer(50, n_sigma_z=3),
                                  Resonator(1e6, 1e9, 1, 1., 1., 0., 0., True))
        return jobs
    seen = _check_batch(make, [9], monkeypatch)
    assert [v for k, v in seen if k == "phx_batch_create"] == created
