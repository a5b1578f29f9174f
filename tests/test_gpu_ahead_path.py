"""Which launch sequence the library takes (phx_engine_three_launch,
phx_batch_three_launch) for the maps, sizes, grids and slicers on which
three-launch and four-launch turns are compared, and where it must keep to
four launches."""
import ctypes as C

import numpy as np
import pytest

from oracle import workloads as W
from tests.machines import COORDS, nonlinear_machine, to_numpy, to_product
from tests.test_gpu_ahead import _map

pytestmark = pytest.mark.gpu


def _three(eng, n_turns):
    from pyheadtail_amd import _phx
    return _phx.lib().phx_engine_three_launch(C.byref(eng._engine), n_turns)


def _paths(make, n, turns, grid=0, rec=False):
    from pyheadtail_amd.engine import FusedOneTurnMap
    b = to_product(W.nonlinear_bunch(n, seed=n))
    eng = FusedOneTurnMap(make(), pass_grid=grid, record_stats=rec, graph_turns=4)
    out = []
    for k in turns:
        eng.track_turns(b, k)
        out.append(_three(eng, k))
    return out, eng


@pytest.mark.parametrize("n", [1, 2, 255, 256, 513, 1024, 131072, 131073, 262657, 500001])
def test_sizes(n):
    print("\n[case] path, n=%d" % n, flush=True)
    assert _paths(lambda: nonlinear_machine(n_slices=37), n, [7, 4, 3, 1])[0] == [1, 1, 0, 0]


@pytest.mark.parametrize("kind", ['rf2/', 'lin/plates', 't_rf/', 'generic/plates', 't/',
                                  'lin/wall'])
@pytest.mark.parametrize("rec", [False, True])
def test_maps(kind, rec):
    print("\n[case] path, %s rec=%s" % (kind, rec), flush=True)
    assert _paths(_map(kind, memory=3), 20011, [5, 1, 9], 768, rec)[0] == [1, 0, 1]


@pytest.mark.parametrize("grid", [1, 5, 300, 768, 2048])
@pytest.mark.parametrize("slicer", [dict(n_sigma_z=2), dict(z_cuts=(-0.3, 0.2)), dict()])
def test_grids_and_cuts(grid, slicer):
    print("\n[case] path, grid %d %r" % (grid, slicer), flush=True)
    assert _paths(_map('lin/', 101, slicer), 60000, [5], grid)[0] == [1]


def test_where_it_stays_at_four_launches(monkeypatch):
    """Tables beyond the LDS (4000 slices), whose results are those of an
    engine that never asked for three launches; a kick on dp."""
    print("\n[case] path, 4000 slices and a longitudinal kick", flush=True)
    from pyheadtail_amd.engine import FusedOneTurnMap
    from pyheadtail_amd.impedances.wakes import Resonator, WakeField
    from pyheadtail_amd.particles.slicing import UniformBinSlicer
    paths, eng = _paths(_map('lin/', 4000), 20000, [8])
    assert paths == [0] and eng._engine.ahead == 1
    record, outs = FusedOneTurnMap._engine_record, []
    for ahead in (True, False):
        with monkeypatch.context() as m:
            m.setattr(FusedOneTurnMap, '_engine_record',
                      lambda self, beam, b, steady: record(self, beam, b, steady and ahead))
            b = to_product(W.nonlinear_bunch(20000, seed=8))
            FusedOneTurnMap(_map('lin/', 4000)(), graph_turns=4).track_turns(b, 8)
            outs.append(to_numpy(b))
    for k in COORDS:
        np.testing.assert_array_equal(outs[0][k], outs[1][k], err_msg=k)

    def longitudinal():
        return _map('lin/')()[:-1] + [WakeField(UniformBinSlicer(64, n_sigma_z=3),
                                                Resonator(1e6, 1e9, 1, 1., 1., 0., 0., True))]
    assert _paths(longitudinal, 20000, [8])[0] == [0]


@pytest.mark.parametrize("n_slices,three", [(64, 1), (4000, 0)])
def test_batch(n_slices, three):
    print("\n[case] path of a batch, %d slices" % n_slices, flush=True)
    from pyheadtail_amd import _phx
    from pyheadtail_amd.batch import BatchedScan
    jobs = [(_map('lin/', s)(), to_product(W.nonlinear_bunch(n, seed=n)))
            for n, s in ((5000, 64), (20011, n_slices))]
    scan = BatchedScan(jobs, graph_turns=4)
    scan.track_turns(9)
    (grp,) = scan._groups.values()
    L = _phx.lib()
    assert L.phx_batch_three_launch(grp['batch'], 9) == three
    assert L.phx_batch_three_launch(grp['batch'], 3) == 0
