"""phx_slice_accumulate over its launch forms: a chunk per block or large
blocks (the particle counts where they change over and around the large
block's size), every number of terms, centres staged in LDS or read from
memory (1200 slices with 8 terms leave no room).  Coordinates and centres are
small whole numbers, so every sum is a whole number that float64 holds and the
results are equal to plain sums."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

CHUNKS = 256                     # at most a chunk per block up to this many
TERMS = [(0, -1, 0, 0), (0, 0, 1, 1), (0, 1, 1, 1), (1, 1, 0, 1), (2, -1, 1, 0), (2, 5, 1, 0),
         (3, 4, 0, 0), (5, 5, 1, 1)]     # a, b, centre_a, centre_b


def _check(n, S, n_terms, given):
    from pyheadtail_amd import _phx
    print("\n[case] slice blocks: n=%d S=%d terms=%d given=%s" % (n, S, n_terms, given), flush=True)
    L, dev = _phx.lib(), _phx.device()
    rng = np.random.default_rng(n + S + n_terms)
    q = rng.integers(-50, 51, (6, n)).astype(np.float64)
    centres = rng.integers(-50, 51, (6, S)).astype(np.float64)
    q[4] = rng.integers(-2, S + 2, n) + 0.25        # z: some outside [0, S)
    idx = np.floor(q[4]).astype(np.int32)
    inside = (idx >= 0) & (idx < S)
    st = _phx.SliceState()
    st.tail, st.head, st.width, st.n, st.n_slices, st.valid = 0., float(S), 1., n, S, 1
    for i in range(6):
        st.absmax[i] = max(50., np.abs(q[i]).max())
    state = _phx.device_record(st)
    t = [torch.from_numpy(q[i].copy()).to(dev) for i in range(6)]
    tc = [torch.from_numpy(centres[i].copy()).to(dev) for i in range(6)]
    terms = (_phx.Term * max(1, n_terms))()
    want = np.zeros((max(1, n_terms), S))
    for k, (a, b, ca, cb) in enumerate(TERMS[:n_terms]):
        terms[k].a, terms[k].b = a, b
        terms[k].center_a = tc[a].data_ptr() if ca else None
        terms[k].center_b = tc[b].data_ptr() if cb and b >= 0 else None
        s = np.where(inside, idx, 0)
        u = q[a] - (centres[a][s] if ca else 0.)
        if b >= 0:
            u = u * (q[b] - (centres[b][s] if cb else 0.))
        want[k] = np.bincount(idx[inside], weights=u[inside], minlength=S)
    gidx = torch.from_numpy(idx).to(dev)
    out = torch.empty(n, dtype=torch.int32, device=dev)
    counts = torch.empty(S, dtype=torch.int32, device=dev)
    sums = torch.full((max(1, n_terms), S), np.nan, dtype=torch.float64, device=dev)
    means = torch.full_like(sums, np.nan)
    ws = _phx.workspace(n, S)
    _phx.call(L.phx_slice_accumulate, _phx.ptr6(t), n, state.data_ptr(), S, terms, n_terms,
              gidx.data_ptr() if given else None, out.data_ptr(), counts.data_ptr(),
              sums.data_ptr(), means.data_ptr(), ws.data_ptr(), _phx.stream())
    ref = np.bincount(idx[inside], minlength=S)
    assert np.array_equal(out.cpu().numpy(), idx)
    assert np.array_equal(counts.cpu().numpy(), ref)
    if n_terms:
        assert np.array_equal(sums.cpu().numpy(), want)
        assert np.array_equal(means.cpu().numpy(), np.where(ref, want / np.maximum(ref, 1), 0.))


@pytest.mark.parametrize("given", [False, True])
@pytest.mark.parametrize("n_terms", range(9))
def test_terms(n_terms, given):
    _check(20011, 100, n_terms, given)


@pytest.mark.parametrize("extra", [-1, 0, 1, 1023, 1024 * 256 + 1])
def test_particle_counts(extra):
    from pyheadtail_amd import _phx
    _check(CHUNKS * _phx.lib().phx_pass_group_size() + extra, 37, 3, False)


@pytest.mark.parametrize("n", [1, 5000, 400000])
def test_centres_beyond_lds(n):
    _check(n, 1200, 8, True)
