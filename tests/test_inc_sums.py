"""The incremental kernel's sums of quantised propensities: integers in
binary64, updated one difference at a time in any order, must stay exact."""

from __future__ import annotations

import re
from pathlib import Path

import numpy as np
import pytest

SOURCE = Path(__file__).resolve().parents[1] / "rebop_amd" / "csrc" / "ssa_inc.hip"


def _window():
    """(lowest, highest, target exponent) of the total, as the kernel has them."""
    text = SOURCE.read_text()
    m = re.search(r"kIncLo = (0x1p\d+), kIncHi = (0x1p\d+);", text)
    t = re.search(r"kIncTarget = (\d+);", text)
    return float.fromhex(m[1]), float.fromhex(m[2]), int(t[1])


@pytest.mark.parametrize("first", ["increases", "decreases", "any"])
def test_a_switch_between_large_propensities_keeps_the_sums_exact(first):
    """Sixteen states, one of them active at a time, with totals over the
    whole upper octave: every event takes away nearly all of the total and
    adds as much elsewhere in the same block of sums."""
    lo, hi, _ = _window()
    rng = np.random.default_rng(5)
    q = [0] * 16
    total = 0.0  # total: the sum as the kernel keeps it
    q[0] = int(rng.integers(int(hi) // 2, int(hi)))
    total += float(q[0])
    for _ in range(20_000):
        new = [int(rng.integers(0, 50)) for _ in q]
        nxt = int(rng.integers(0, 16))
        new[nxt] = int(rng.integers(int(hi) // 2, int(hi) - 1000))
        steps = [float(b - a) for a, b in zip(q, new)]
        if first == "any":
            rng.shuffle(steps)
        else:
            steps.sort(reverse=first == "increases")
        for d in steps:
            total += d
        q = new
        assert lo <= sum(q) < hi
        assert int(total) == sum(q)


def test_a_total_past_the_window_is_never_taken_for_one_inside():
    """Just above the window the additions may lose units; the total found
    must still call for a rebuild."""
    _, hi, _ = _window()
    rng = np.random.default_rng(6)
    for _ in range(20_000):
        old = [int(hi) - 1 - int(rng.integers(0, 4))] + [int(v) for v in rng.integers(0, 2, size=9)]
        old[0] -= sum(old[1:])
        new = [int(v) for v in rng.integers(0, 4, size=9)] + [int(hi) + int(rng.integers(0, 12))]
        total = float(sum(old))
        steps = [float(b - a) for a, b in zip(old, new)]
        if rng.random() < 0.5:
            steps.sort(reverse=True)
        else:
            rng.shuffle(steps)
        for d in steps:
            total += d
        if sum(new) >= hi:
            assert total >= hi


def test_a_rebuild_puts_the_total_well_inside_the_window():
    lo, hi, target = _window()
    # quantisation moves the total by half a unit per reaction, at most 4096
    assert 2.0**target - 4096 > lo and 2.0 ** (target + 1) + 4096 < hi


@pytest.mark.gpu
def test_alternating_large_propensities_bit_exact(nthreads):
    """A switch between two species of very different totals, next to slow
    reactions, over several octaves of the total."""
    from tests.networks import build_device, build_oracle

    import torch

    S, rx = 36, []
    for i in range(16):  # one token walks round, its exit rates 3:1 apart
        o, d = [0] * S, [0] * S
        o[i] = 1
        d[i], d[(i + 1) % 16] = -1, 1
        rx.append((3e5 if i % 2 else 1e5 * (1 + i % 5), o, d))
    for i in range(16, S - 1):
        o, d = [0] * S, [0] * S
        o[i] = 1
        d[i], d[i + 1] = -1, 1
        rx.append((0.7, o, d))
    spec = (S, rx, [1] + [0] * 15 + [3] * (S - 16))
    n, nb, tmax = 24, 9, 0.05
    g = build_device(spec, 4)
    out = torch.zeros((nb + 1, S, n), dtype=torch.int64, device="cuda")
    st = g.run_device(tmax, nb, n, out.data_ptr())
    torch.cuda.synchronize()
    _, oout, _, oev, odr = build_oracle(spec, sparse=True).run_grid(4, spec[2], tmax, nb, n_traj=n, nthreads=nthreads)
    assert np.array_equal(out.cpu().numpy(), oout)
    assert (st.events, st.draws) == (oev, odr) and oev > 100_000
