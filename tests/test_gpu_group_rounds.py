"""GPU parity of the grouped kernels' rounds (several lanes per trajectory),
bit for bit against the CPU oracle, where a round can go wrong: trajectories
that end, or are absorbed, at any of its draws; sample times at and past the
LDS copy's limit; run sizes at which the lanes per trajectory change; runs to
one target time, and runs with every event recorded."""

from __future__ import annotations

import numpy as np
import pytest

from rebop_amd import _native as K
from tests.networks import build_device, build_oracle

pytestmark = pytest.mark.gpu
SPEC = K.REBOP_KERNEL_PLAIN | K.REBOP_KERNEL_SPECIALIZED
KINDS = [K.REBOP_KERNEL_AUTO, SPEC | K.REBOP_KERNEL_GROUP4, SPEC | K.REBOP_KERNEL_GROUP2]

SIR = (3, [(1e-4, [1, 1, 0], [-1, 1, 0]), (0.01, [0, 1, 0], [0, -1, 1])], [999, 1, 0])
# absorbed after exactly `m` events, and never moving at all
DECAY = lambda m: (2, [(1.0, [1, 0], [-1, 1])], [m, 0])  # noqa: E731
# no absorbing state, and one a jump can leave only by another reaction
BIRTH = (2, [(30.0, [0, 0], [1, 0]), (0.5, [1, 0], [-1, 2]), (0.1, [0, 1], [0, -1])], [0, 3])


def _same(spec, tmax, nb, n, kernel, nthreads, seed=23):
    import torch

    g = build_device(spec, seed)
    out = torch.full((nb + 1, spec[0], n + 1), -7, dtype=torch.int64, device="cuda")[:, :, :n].contiguous()
    fin = torch.zeros((spec[0], n), dtype=torch.int64, device="cuda")
    st = g.run_device(tmax, nb, n, out.data_ptr(), final_ptr=fin.data_ptr(), kernel=kernel, traj_begin=5)
    torch.cuda.synchronize()
    _, oout, _, oev, odr = build_oracle(spec).run_grid(seed, spec[2], tmax, nb, n_traj=n, traj_begin=5,
                                                       nthreads=nthreads)
    assert np.array_equal(out.cpu().numpy(), oout)
    assert np.array_equal(fin.cpu().numpy(), oout[nb])
    assert (st.events, st.draws) == (oev, odr)
    return st


@pytest.mark.parametrize("kernel", KINDS)
@pytest.mark.parametrize("m", [0, 1, 2, 3, 4, 5, 15, 16, 17, 33])
def test_absorbed_at_any_draw_of_a_round(m, kernel, nthreads):
    for nb in (1, 6, 31):
        _same(DECAY(m), 3.0, nb, 37, kernel, nthreads)


@pytest.mark.parametrize("kernel", KINDS)
@pytest.mark.parametrize("nb", [1, 3, 2047, 2048])
def test_sample_counts_around_the_lds_copy(nb, kernel, nthreads):
    _same(BIRTH, 2.0, nb, 19, kernel, nthreads)


@pytest.mark.parametrize("n", [1, 4, 15, 17, 4095, 4097])
def test_run_sizes_where_the_lanes_change(n, nthreads):
    st = _same(SIR, 60.0, 7, n, K.REBOP_KERNEL_AUTO, nthreads)
    assert st.kernel & K.REBOP_KERNEL_GROUP4


@pytest.mark.parametrize("n", [1, 63, 4100])
@pytest.mark.parametrize("spec", [SIR, DECAY(9), BIRTH])
def test_targets(spec, n):
    """A batch advanced twice, against the oracle's single trajectories."""
    b = build_device(spec, 23).batch(n, traj_begin=5)
    o = build_oracle(spec)
    some = sorted({0, n // 2, n - 1, *range(0, n, 331)})
    want = [o.state(spec[2], 23, traj=5 + j) for j in some]
    for target in (1.5, 40.0):
        b.advance_until(target)
        x, t, draws = b.get_species(), b.get_time(), b.get_draws()
        for j, w in zip(some, want):
            w.advance_until(target)
            assert np.array_equal(x[j], w.x) and t[j] == w.t and draws[j] == w.draws, (j, target)


@pytest.mark.parametrize("n", [2, 19, 300])
@pytest.mark.parametrize("spec,tmax", [(SIR, 60.0), (DECAY(0), 3.0), (DECAY(1), 30.0), (DECAY(7), 30.0), (BIRTH, 2.0)])
def test_every_event_recorded(spec, tmax, n):
    ts, xs = build_device(spec, 23).run_all_events(tmax, n_traj=n, traj_begin=5)
    o = build_oracle(spec)
    for j in range(n):
        t, x = o.run_all_events(23, 5 + j, spec[2], tmax)
        assert np.array_equal(ts[j].view(np.uint64), t.view(np.uint64)) and np.array_equal(xs[j], x), j


@pytest.mark.parametrize("n", [3, 64, 4100, 40_000])
def test_a_time_set_to_nan_fires_until_absorbed(n):
    """No sample time is before NaN, so such a trajectory runs on to its
    absorbing state, whatever the lanes per trajectory (16, 4, 2, 1)."""
    b = build_device(DECAY(9), 23).batch(n, traj_begin=5)
    t = np.zeros(n)
    t[::3] = np.nan
    b.set_time(t)
    b.advance_until(0.7)
    x, time, draws = b.get_species(), b.get_time(), b.get_draws()
    assert np.array_equal(x[::3], np.tile([0, 9], (len(x[::3]), 1)))
    assert np.array_equal(draws[::3], np.full(len(draws[::3]), 9))
    assert np.array_equal(time, np.full(n, 0.7))
    o = build_oracle(DECAY(9))
    for j in range(1, min(n, 60), 3):  # the others of the same waves
        w = o.state(DECAY(9)[2], 23, traj=5 + j)
        w.advance_until(0.7)
        assert np.array_equal(x[j], w.x) and draws[j] == w.draws, j
