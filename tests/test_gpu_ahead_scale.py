"""Three-launch turns scale a turn's slice sums by the largest |x| of the state
before the turn, four-launch turns by that after it.  The scale is a power of
2^8, so the sums are equal unless the two straddle a step; there each side
keeps a value to half a unit of 2^(P - 73), P the exponent of its scale.  Here
the largest |x| crosses 2^-9 (P = 0 above, -8 below) in the turn compared, in
slices of one macroparticle, some of them with |x| of a few nanometres."""
import numpy as np
import pytest

from oracle import workloads as W

pytestmark = pytest.mark.gpu

TURN = 5


def _run(q, ahead, monkeypatch):
    from pyheadtail_amd.engine import FusedOneTurnMap
    from pyheadtail_amd.impedances.wakes import CircularResonator, WakeField
    from pyheadtail_amd.particles.particles import Particles
    from pyheadtail_amd.particles.slicing import UniformBinSlicer
    from tests.machines import linear_machine
    record = FusedOneTurnMap._engine_record
    n = len(q["x"])
    b = Particles(n, 1e-6, W.e, W.m_p, W.CIRCUMFERENCE, W.GAMMA, q)
    wake = WakeField(UniformBinSlicer(4 * n, z_cuts=(-0.3, 0.3)), CircularResonator(1e6, 1e9, 1))
    with monkeypatch.context() as m:
        m.setattr(FusedOneTurnMap, "_engine_record",
                  lambda self, beam, b, steady: record(self, beam, b, steady and ahead))
        eng = FusedOneTurnMap(linear_machine() + [wake], graph_turns=0)
        eng.track_turns(b, TURN)
    _, counts, mean_x, _ = eng.slice_data
    return counts.cpu().numpy(), mean_x.cpu().numpy(), np.abs(b.x.cpu().numpy()).max()


def test_scale_step_between_two_states(monkeypatch):
    print("\n[case] largest |x| crosses a scale step", flush=True)
    n = 200                       # every particle counts for the largest |x|
    rng = np.random.default_rng(2)
    q = {k: np.zeros(n) for k in ("x", "xp", "y", "yp", "z", "dp")}
    q["x"] = rng.uniform(-1., 1., n) * 1e-9
    q["x"][0] = 2e-3
    q["z"] = np.linspace(-0.25, 0.25, n)
    # particle 0's |x| after t turns is |cos| of t times the tune
    peak = [2e-3 * abs(np.cos(2 * np.pi * W.Q_X * t)) for t in (TURN - 1, TURN)]
    q["x"] *= 2.**-9 / np.sqrt(peak[0] * peak[1])
    counts, three, last = _run(q, True, monkeypatch)
    counts4, four, _ = _run(q, False, monkeypatch)
    before = last * peak[0] / peak[1]
    assert min(before, last) < 0.99 * 2.**-9 and max(before, last) > 1.01 * 2.**-9
    np.testing.assert_array_equal(counts, counts4)
    assert counts.max() == 1 and counts.sum() == n
    # half a unit at P = 0 and at P = -8, and the rounding of a mean (below 2^-62)
    tol = 2.**-74 + 2.**-82 + np.spacing(np.abs(four))
    assert np.all(np.abs(three - four) <= tol)
    assert np.any(three != four)
