"""GPU parity of the incremental kernel (AUTO's choice for large networks and
job batches) against the CPU oracle, bit for bit."""

from __future__ import annotations

import numpy as np
import pytest

from rebop_amd import _native, expr, workloads
from rebop_amd.engine import GillespieNet, Rate, RateExpr, run_jobs
from tests.networks import build_device, build_oracle, synthetic

pytestmark = pytest.mark.gpu
AUTO = _native.REBOP_KERNEL_AUTO
LDS = _native.REBOP_KERNEL_LDS


def _run(g, tmax, nb, n, x0=None, traj_begin=0, stats=True):
    import torch

    S = g.nb_species()
    out = torch.zeros((nb + 1, S, n), dtype=torch.int64, device="cuda")
    fin = torch.zeros((S, n), dtype=torch.int64, device="cuda")
    xt = None if x0 is None else torch.as_tensor(np.ascontiguousarray(x0, dtype=np.int64), device="cuda")
    st = g.run_device(tmax, nb, n, out.data_ptr(), x0_ptr=None if xt is None else xt.data_ptr(),
                      final_ptr=fin.data_ptr(), traj_begin=traj_begin, kernel=AUTO, with_stats=stats)
    torch.cuda.synchronize()
    out = out.cpu().numpy()
    assert np.array_equal(out[-1], fin.cpu().numpy())
    return out, st


def _check(g, o, x0, tmax, nb, n, seed, nthreads, traj_begin=0, per_traj=None):
    out, st = _run(g, tmax, nb, n, x0=per_traj, traj_begin=traj_begin)
    assert st.kernel & 0xF == LDS
    _, oout, _, oev, odr = o.run_grid(seed, x0 if per_traj is None else per_traj, tmax, nb, n_traj=n,
                                      traj_begin=traj_begin, x0_per_traj=per_traj is not None,
                                      nthreads=nthreads)
    assert np.array_equal(out, oout), np.argwhere(out != oout)[:5].tolist()
    assert (st.events, st.draws, st.trajectories) == (oev, odr, n)
    return oout, oev


# blocks hold 8 reactions up to 512, then 16, 32, ...; super-blocks 64 each;
# a wave holds 8 trajectories
@pytest.mark.parametrize("S,R,n", [(33, 1, 3), (33, 7, 8), (40, 8, 9), (40, 9, 1), (33, 63, 65), (33, 64, 64),
                                   (33, 65, 130), (33, 512, 20), (100, 513, 17), (64, 1030, 9), (250, 300, 16),
                                   (40, 2100, 8)])
def test_sizes_bit_exact(S, R, n, nthreads):
    spec = synthetic(S, R, 100 + R, init_mean=40.0, bounded=True)
    total = workloads.initial_total_propensity(spec)
    _check(build_device(spec, 9), build_oracle(spec, sparse=True), spec[2], 300.0 / total if total else 1.0, 11,
           n, 9, nthreads, traj_begin=5)


def test_per_trajectory_counts(nthreads):
    """Initial counts per trajectory, among them empty (absorbing) and
    negative ones (a negative propensity: the reference's own sums)."""
    spec = synthetic(40, 90, 4, init_mean=30.0, bounded=True)
    x0 = np.random.default_rng(1).poisson(30.0, size=(41, 40)).astype(np.int64)
    x0[3] = 0
    x0[7, ::3] = -2
    x0[11, 5] = -1
    _check(build_device(spec, 21), build_oracle(spec, sparse=True), None, 0.02, 9, 41, 21, nthreads, per_traj=x0)


def _expr_net(S, rx, x0, seed):
    """Device and oracle network; rx: (rate or expression text, orders, diffs)."""
    from oracle.pyoracle import OracleNet

    names = {f"X{i}": i for i in range(S)}
    g, o = GillespieNet(x0, seed=seed), OracleNet(S)
    for rate, orders, d in rx:
        if isinstance(rate, str):
            code, consts = expr.to_postfix(expr.parse(rate), names, {})
            g.add_reaction(RateExpr.from_postfix(code, consts), d)
            o.add_expr(code, consts, d)
        else:
            g.add_reaction(Rate.lma(rate, orders), d)
            o.add_lma(rate, orders, d)
    return g, o


def test_expressions_that_go_negative(nthreads):
    """Propensities and counts below zero: the sums are no longer monotone
    and the choice counts every smaller partial sum."""
    S = 40
    rx = []
    for i in range(S):
        d = [0] * S
        d[i], d[(i + 1) % S] = -1, 1
        text = [f"0.1 * X{i} - 1.5", f"2 * X{i} / (1 + X{(i + 3) % S} ^ 2)", f"max(X{i}, 1) * exp(-X{i} / 9)",
                f"min(X{i}, 3) * -(X{(i + 5) % S} - 20) / 40", f"0.2 * X{i}"][i % 5]
        rx.append((text, None, d))
    x0 = [12 + (7 * i) % 9 for i in range(S)]
    g, o = _expr_net(S, rx, x0, 31)
    oout, oev = _check(g, o, x0, 9.0, 20, 50, 31, nthreads)
    assert oout.min() < 0 and oev > 50 * 20


def test_long_jumps_and_small_totals(nthreads):
    """Jumps beyond the update list's 8 bits, and a total that falls by many
    powers of two (the sums' unit moves) down to an absorbing state."""
    S = 34
    rx = []
    for i in range(S - 1):
        o, d = [0] * S, [0] * S
        o[i] = 1
        d[i] = -1
        d[i + 1] = 1 if i else 300
        rx.append((10.0 ** (3 - 0.4 * i), o, d))
    spec = (S, rx, [7] + [5] * (S - 1))
    oout, _ = _check(build_device(spec, 2), build_oracle(spec, sparse=True), spec[2], 1e12, 30, 40, 2, nthreads)
    assert oout[-1].min() == 0 and oout[-1, -1].min() > 300  # all in the last species


def test_sample_time_equal_to_an_event_time(nthreads):
    """A sample time that an event hits exactly: the time interval straddles
    it and the trajectory is decided by the reference's own sums."""
    spec = synthetic(40, 120, 8, init_mean=30.0, bounded=True)
    o = build_oracle(spec, sparse=True)
    for traj, event in ((0, 5), (3, 60), (6, 200)):
        times, _ = o.run_all_events(17, traj, spec[2], 0.05)[:2]
        _check(build_device(spec, 17), o, spec[2], float(times[event]), 1, 10, 17, nthreads)


def test_choice_on_a_boundary(nthreads):
    """Propensities chosen so that trajectory 4's first threshold falls on a
    partial sum: within the sums' rounding, so the choice is the reference's."""
    from oracle import pyoracle

    w = pyoracle.stream_block(23, 4, 0)
    u = ((int(w[3]) << 32 | int(w[2])) >> 11) * 2.0**-53
    S = 40
    for step in (-1, 0, 1):
        k0 = u / (1.0 - u)
        k0 = float(np.nextafter(k0, k0 + step)) if step else k0
        rx = []
        for i, k in ((0, k0), (1, 1.0)):
            orders, d = [0] * S, [0] * S
            orders[i] = 1
            d[i], d[2 + i] = -1, 1
            rx.append((k, orders, d))
        spec = (S, rx, [1, 1] + [0] * (S - 2))
        _check(build_device(spec, 23), build_oracle(spec, sparse=True), spec[2], 1.0, 4, 8, 23, nthreads)


def test_counts_beyond_int32_rerun_and_async(nthreads):
    """A count that passes 2^30: rerun with int64 counts; with no counters to
    read, the trajectories that stay in range are right."""
    S = 40
    rx = [(2.0, [0] * S, [2**20] + [0] * (S - 1)), (2e-9, [1] + [0] * (S - 1), [-1, 1] + [0] * (S - 2))]
    for i in range(2, S - 1):
        o, d = [0] * S, [0] * S
        o[i], d[i], d[i + 1] = 1, -1, 1
        rx.append((0.3, o, d))
    spec = (S, rx, [2**30 - 3 * 2**20, 0] + [20] * (S - 2))
    oout, _ = _check(build_device(spec, 8), build_oracle(spec, sparse=True), spec[2], 6.0, 12, 40, 8, nthreads)
    assert oout.max() > 2**30
    x0 = np.tile(np.asarray(spec[2], dtype=np.int64), (24, 1))
    x0[:12, 0] = 100
    out, st = _run(build_device(spec, 8), 6.0, 12, 24, x0=x0, stats=False)
    assert st is None
    _, oout, _, _, _ = build_oracle(spec, sparse=True).run_grid(8, x0[:12], 6.0, 12, n_traj=12, x0_per_traj=True,
                                                                nthreads=nthreads)
    assert np.array_equal(out[:, :, :12], oout)


def test_job_batch_of_many_shapes(nthreads):
    """One launch of networks of 3 to 600 reactions, one with expressions."""
    import torch

    specs = [synthetic(3 + 4 * i, r, 50 + r, init_mean=30.0, bounded=True)
             for i, r in enumerate((3, 8, 17, 64, 129, 300, 600))]
    nets = [(build_device(s, 3), build_oracle(s, sparse=True), s[2]) for s in specs]
    rx = [("3 / (1 + (X1 / 4)^2)", None, [1, 0]), ("exp(-X0 / 8) * X0", None, [-1, 1]), (0.5, [0, 1], [0, -1])]
    nets.append((*_expr_net(2, rx, [5, 0], 3), [5, 0]))
    sizes = [70, 1, 8, 33, 9, 16, 5, 40]
    horizon = [0.05] * 7 + [10.0]
    bufs = [torch.zeros((7, len(x), n), dtype=torch.int64, device="cuda") for (_, _, x), n in zip(nets, sizes)]
    st, ev = run_jobs([dict(net=g, tmax=t, nb_steps=6, n_traj=n, traj_begin=i, out_ptr=b.data_ptr())
                       for i, ((g, _, _), n, t, b) in enumerate(zip(nets, sizes, horizon, bufs))],
                      per_job_events=True)
    torch.cuda.synchronize()
    assert st.trajectories == sum(sizes) and st.events == int(ev.sum())
    for i, ((_, o, x), n, t, b) in enumerate(zip(nets, sizes, horizon, bufs)):
        _, oout, _, oev, _ = o.run_grid(3, x, t, 6, n_traj=n, traj_begin=i, nthreads=nthreads)
        assert np.array_equal(b.cpu().numpy(), oout), i
        assert int(ev[i]) == oev
