"""Three-launch turns of the two-harmonic orders against the four-launch turns,
bit for bit, with the detuner sets that take two and three groups of threads a
block, at the particle counts where a block's groups are partly or all used."""
import numpy as np
import pytest

from oracle import workloads as W
from tests.machines import smooth_transverse
from tests.test_gpu_ahead import _check, _map

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first", ["rf", "segment"])
@pytest.mark.parametrize("amplitude", [False, True])
@pytest.mark.parametrize("n,grid", [(1, 0), (1025, 0), (300001, 0), (60000, 300), (60000, 5)])
def test_two_harmonics(first, amplitude, n, grid, monkeypatch):
    print("\n[case] two harmonics, %s first, amplitude %s, n=%d grid=%d"
          % (first, amplitude, n, grid), flush=True)
    rf, _, wake = _map('rf2/')()
    app = 1e-10 * W.P0 if amplitude else 0.

    def make():
        seg = smooth_transverse(5., app, -0.5 * app)[0]
        return ([rf, seg] if first == "rf" else [seg, rf]) + [wake]
    _check(make, W.nonlinear_bunch(n, seed=n), [6], monkeypatch, grid=grid)
