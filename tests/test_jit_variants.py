"""Which kernels a network's run-time compilation holds: those of the run
that is made (or, prepared, those of a grid run of any size), not all of them."""

from __future__ import annotations

import re

import numpy as np
import pytest

from rebop_amd import _native
from rebop_amd.engine import GillespieNet, Rate
from tests.networks import build_device, build_oracle, sir, synthetic


@pytest.fixture
def kernels(tmp_path, monkeypatch):
    """The entry points of the module that was compiled since the last call."""
    dump = tmp_path / "kernel.hip"
    monkeypatch.setenv("REBOP_DUMP_SPECIALIZED", str(dump))
    monkeypatch.setenv("REBOP_JIT_CACHE", "")

    def names():
        if not dump.exists():
            return set()
        text = dump.read_text()
        dump.unlink()
        return set(re.findall(r'extern "C" __global__ .*?rebop_ssa_jit_(\w+)\(', text))

    return names


@pytest.mark.parametrize("spec,lanes", [(sir(), {"g16"}), (synthetic(6, 32, 2), {"g16"}), (synthetic(6, 33, 2), set())])
def test_prepared_for_grid_runs_of_any_size(spec, lanes, kernels):
    g = build_device(spec, 90 + len(spec[1]))
    g.prepare()
    assert kernels() == {"main", "g2", "g4", "g2_far", "g4_far"} | lanes


def test_prepared_with_a_draw_cap(kernels):
    g = build_device(sir(), 91)
    g.set_draw_cap(50_000)
    g.prepare()
    assert kernels() - {"g16"} == {"main", "g2", "g4", "g2_far", "g4_far"}  # (with a device, without the cap too)


def _fresh(k):
    """A network no other test compiles."""
    g = GillespieNet([40, 3, 0], seed=12)
    g.add_reaction(Rate.lma(1e-3 * (1 + k / 97), [1, 1, 0]), [-1, 1, 0])
    g.add_reaction(Rate.lma(0.25, [0, 1, 0]), [0, -1, 1])
    return g, (3, [(1e-3 * (1 + k / 97), [1, 1, 0], [-1, 1, 0]), (0.25, [0, 1, 0], [0, -1, 1])], [40, 3, 0])


def _grid(g, spec, n, nthreads):
    import torch

    out = torch.zeros((6, 3, n), dtype=torch.int64, device="cuda")
    g.run_device(8.0, 5, n, out.data_ptr())
    torch.cuda.synchronize()
    _, oout, _, _, _ = build_oracle(spec).run_grid(12, spec[2], 8.0, 5, n_traj=n, nthreads=nthreads)
    assert np.array_equal(out.cpu().numpy(), oout)


@pytest.mark.gpu
def test_a_run_compiles_what_it_launches(kernels, nthreads):
    g, spec = _fresh(1)
    for n, want in ((100, {"g16"}), (200, set()), (5000, {"g4"}), (40_000, {"main"}), (20_000, {"g2"}),
                    (30, set())):
        _grid(g, spec, n, nthreads)
        assert kernels() == want, n
    g.prepare()
    assert kernels() == {"g2_far", "g4_far"}  # for more sample times than LDS holds


@pytest.mark.gpu
def test_the_tail_comes_with_the_main_kernel(kernels, nthreads):
    g, spec = _fresh(2)
    _grid(g, spec, 40_000, nthreads)
    assert kernels() == {"main", "g4"}
    other, spec2 = _fresh(2)  # another handle of the same network: nothing to compile
    _grid(other, spec2, 33_000, nthreads)
    assert kernels() == set()


@pytest.mark.gpu
def test_every_event_recorded_and_sweeps(kernels):
    import torch

    g, spec = _fresh(3)
    o = build_oracle(spec)
    ts, xs = g.run_all_events(8.0, n_traj=20)
    assert kernels() == {"ev4_write"}  # the counting pass before it: ev4_count, compiled first
    for j in (0, 7, 19):
        t, x = o.run_all_events(12, j, spec[2], 8.0)
        assert np.array_equal(ts[j], t) and np.array_equal(xs[j], x)
    out = torch.zeros((4, 3, 6), dtype=torch.int64, device="cuda")
    rates = torch.tensor([[spec[1][0][0], 0.25]] * 2, dtype=torch.float64, device="cuda")
    g.run_sweep_device(2, 3, 8.0, 3, out.data_ptr(), rates_ptr=rates.data_ptr())
    torch.cuda.synchronize()
    assert kernels() == {"sweep"}
    _, oout, _, _, _ = o.run_grid(12, spec[2], 8.0, 3, n_traj=6)
    assert np.array_equal(out.cpu().numpy(), oout)


@pytest.mark.gpu
def test_a_prepared_module_on_disk_serves_single_variants(tmp_path, monkeypatch, nthreads):
    """The disk cache holds the prepared module: a handle on it compiles
    nothing (its own in-process module aside, which this network has not)."""
    monkeypatch.setenv("REBOP_JIT_CACHE", str(tmp_path / "co"))
    g, spec = _fresh(4)
    g.prepare()
    before = sorted((tmp_path / "co").iterdir())
    assert len(before) == 2  # one module and its source
    for n in (50, 5000, 40_000):
        _grid(g, spec, n, nthreads)
    assert sorted((tmp_path / "co").iterdir()) == before


# networks on both sides of the limit for 16 lanes
@pytest.mark.gpu
@pytest.mark.parametrize("S,R", [(5, 32), (5, 33), (32, 64)])
def test_larger_networks_in_grouped_rounds(S, R, nthreads):
    import torch

    spec = synthetic(S, R, 60 + R, init_mean=12.0, bounded=True)
    o = build_oracle(spec)
    SPEC = _native.REBOP_KERNEL_PLAIN | _native.REBOP_KERNEL_SPECIALIZED
    for kernel in (_native.REBOP_KERNEL_AUTO, SPEC | _native.REBOP_KERNEL_GROUP4, SPEC | _native.REBOP_KERNEL_GROUP2):
        for nb, n in ((7, 37), (2048, 5)):  # straight rounds, and step by step
            out = torch.zeros((nb + 1, S, n), dtype=torch.int64, device="cuda")
            st = build_device(spec, 6).run_device(0.5, nb, n, out.data_ptr(), kernel=kernel)
            torch.cuda.synchronize()
            _, oout, _, oev, odr = o.run_grid(6, spec[2], 0.5, nb, n_traj=n, nthreads=nthreads)
            assert np.array_equal(out.cpu().numpy(), oout), (kernel, nb)
            assert (st.events, st.draws) == (oev, odr)
    ts, xs = build_device(spec, 6).run_all_events(0.5, n_traj=9)
    for j in range(9):
        t, x = o.run_all_events(6, j, spec[2], 0.5)
        assert np.array_equal(ts[j].view(np.uint64), t.view(np.uint64)) and np.array_equal(xs[j], x), j
