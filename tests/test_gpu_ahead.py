"""Three-launch turns (the pass slices its own turn and sums the next turn's z)
against the four-launch turns of the same engine: coordinates, slices, kicks
and statistics bit for bit, at the edges of groups and grids, for every cuts
mode, and where the fixed-point scale of the slices' sums comes from a state
that says little about the next one."""
import numpy as np
import pytest

from oracle import workloads as W
from tests.machines import COORDS, nonlinear_machine, smooth_transverse, to_numpy, to_product

pytestmark = pytest.mark.gpu


def _run(make, ob, turns, ahead, monkeypatch, grid=0, rec=False, graph=0, change=None):
    from pyheadtail_amd.engine import FusedOneTurnMap
    record = FusedOneTurnMap._engine_record

    def patched(self, beam, b, steady):
        return record(self, beam, b, steady and ahead)
    with monkeypatch.context() as m:
        m.setattr(FusedOneTurnMap, '_engine_record', patched)
        b = to_product(ob)
        if change is not None:
            change(b)
        eng = FusedOneTurnMap(make(), pass_grid=grid, record_stats=rec, graph_turns=graph)
        for k in turns:
            eng.track_turns(b, k)
        assert eng._engine.ahead == (1 if ahead else 0)
        out = to_numpy(b)
    z_bins, counts, mx, my = eng.slice_data
    out.update(z_bins=z_bins.cpu().numpy(), counts=counts.cpu().numpy(), mx=mx.cpu().numpy(),
               my=my.cpu().numpy(), kicks=eng.pending_kicks.cpu().numpy())
    if rec:
        out['stats'] = eng.last_stats['raw']
    return out


def _check(make, ob, turns, monkeypatch, **kw):
    a = _run(make, ob, turns, True, monkeypatch, **kw)
    b = _run(make, ob, turns, False, monkeypatch, **kw)
    for k in a:
        np.testing.assert_array_equal(a[k], b[k], err_msg=k)
    return a


def _map(kind, n_slices=64, slicer_kw=None, memory=1):
    from scipy.constants import e, m_p
    from pyheadtail_amd.impedances.wakes import (CircularResonator, WakeField,
                                                 ParallelHorizontalPlatesResistiveWall,
                                                 ParallelHorizontalPlatesResonator)
    from pyheadtail_amd.particles.slicing import UniformBinSlicer
    from pyheadtail_amd.trackers.longitudinal_tracking import LinearMap, RFSystems

    def rf(nh):
        return RFSystems(W.CIRCUMFERENCE, [W.H_RF, 4 * W.H_RF][:nh], [W.V_RF, 0.1 * W.V_RF][:nh],
                         [0.2, np.pi][:nh], [W.ALPHA_C], W.GAMMA, p_increment=0., charge=e,
                         mass=m_p)
    seg = smooth_transverse(5., 1e-10 * W.P0, -5e-11 * W.P0)[0]
    lin = LinearMap(np.atleast_1d(W.ALPHA_C), W.CIRCUMFERENCE, 0.017)
    src = {'plates': ParallelHorizontalPlatesResonator(1e6, 1e9, 1),
           'wall': ParallelHorizontalPlatesResistiveWall(0.02, W.CIRCUMFERENCE, 5.9e7, 1e-12,
                                                         n_turns_wake=memory)}
    els = {'rf2': [rf(2), seg], 'lin': [lin, seg], 't_rf': [seg, rf(1)],
           'generic': [seg, lin, smooth_transverse(3.)[0]], 't': [seg]}
    el, _, wk = kind.partition('/')
    sl = UniformBinSlicer(n_slices, **(slicer_kw or dict(n_sigma_z=3)))
    return lambda: els[el] + [WakeField(sl, src.get(wk, CircularResonator(1e6, 1e9, 1)))]


@pytest.mark.parametrize("n", [1, 2, 255, 256, 513, 1024, 131072, 131073, 262657, 500001])
def test_sizes(n, monkeypatch):
    print("\n[case] three-launch turns, n=%d" % n, flush=True)
    _check(lambda: nonlinear_machine(n_slices=37), W.nonlinear_bunch(n, seed=n), [7], monkeypatch)


@pytest.mark.parametrize("kind", ['rf2/', 'lin/plates', 't_rf/', 'generic/plates', 't/',
                                  'lin/wall'])
@pytest.mark.parametrize("rec", [False, True])
def test_maps_and_statistics(kind, rec, monkeypatch):
    print("\n[case] three-launch turns, %s rec=%s" % (kind, rec), flush=True)
    _check(_map(kind, memory=3), W.nonlinear_bunch(20011, seed=5), [5, 1, 9], monkeypatch, rec=rec,
           graph=4, grid=768)


@pytest.mark.parametrize("grid", [1, 5, 300, 768, 2048])
@pytest.mark.parametrize("slicer", [dict(n_sigma_z=2), dict(z_cuts=(-0.3, 0.2)), dict()])
def test_grids_and_cuts(grid, slicer, monkeypatch):
    print("\n[case] three-launch turns, grid %d %r" % (grid, slicer), flush=True)
    _check(_map('lin/', 101, slicer), W.nonlinear_bunch(60000, seed=6), [5], monkeypatch, grid=grid)


@pytest.mark.parametrize("kind", ["zero_x", "halo", "nan_z", "nan_x", "shifted_z"])
def test_scales_and_non_finite_values(kind, monkeypatch):
    """zero_x: the first turn's bound of |x| is zero; halo: a few particles far
    beyond the bound that the sampled ones give; NaN particles."""
    print("\n[case] three-launch turns, %s" % kind, flush=True)

    def change(b):
        if kind == "zero_x":
            b.x.zero_()
        elif kind == "halo":
            b.x[7000:7004] *= 1e5
        elif kind == "nan_z":
            b.z[123] = float("nan")
        elif kind == "nan_x":
            b.x[123] = float("nan")
        else:
            b.z += 1e-3
    slicer = dict(z_cuts=(-0.5, 0.5)) if kind.startswith("nan") else None
    out = _check(_map('lin/', 50, slicer), W.nonlinear_bunch(30001, seed=7), [5, 4], monkeypatch,
                 change=change)
    if kind == "nan_z":
        assert np.isfinite(out['mx']).all()


def test_many_slices_keep_the_four_launch_turn():
    """A histogram and kick table beyond the LDS: four-launch turns."""
    print("\n[case] 4000 slices", flush=True)
    ob = W.nonlinear_bunch(20000, seed=8)
    from pyheadtail_amd.engine import FusedOneTurnMap
    outs = []
    for graph in (0, 4):
        b = to_product(ob)
        FusedOneTurnMap(_map('lin/', 4000)(), graph_turns=graph).track_turns(b, 8)
        outs.append(to_numpy(b))
    for k in COORDS:
        np.testing.assert_array_equal(outs[0][k], outs[1][k], err_msg=k)
