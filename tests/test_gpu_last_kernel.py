"""Which kernel a run took (rebop_last_kernel): the parity tests elsewhere
compare results that every kernel gives, so here each way through the dispatch
is named."""

from __future__ import annotations

import numpy as np
import pytest

from rebop_amd import _native as K
from rebop_amd import workloads
from rebop_amd.engine import run_jobs
from tests.networks import build_device, build_oracle, dimers, sir, synthetic
from tests.test_gpu_inc import _expr_net

pytestmark = pytest.mark.gpu
AUTO, SPEC = K.REBOP_KERNEL_AUTO, K.REBOP_KERNEL_PLAIN | K.REBOP_KERNEL_SPECIALIZED
PERSISTENT = K.REBOP_KERNEL_PERSISTENT | K.REBOP_KERNEL_SPECIALIZED


def _run(g, n, tmax=0.01, nb=4, kernel=AUTO):
    import torch

    out = torch.empty((nb + 1, g.nb_species(), n), dtype=torch.int64, device="cuda")
    st = g.run_device(tmax, nb, n, out.data_ptr(), kernel=kernel)
    torch.cuda.synchronize()
    return K.last_kernel(), out, st


# the sizes of the incremental kernel's parity tests
@pytest.mark.parametrize("S,R,n", [(33, 1, 3), (33, 7, 8), (40, 8, 9), (40, 9, 1), (33, 63, 65), (33, 64, 64),
                                   (33, 65, 130), (33, 512, 20), (100, 513, 17), (64, 1030, 9), (250, 300, 16),
                                   (40, 2100, 8)])
def test_large_networks_take_the_incremental_kernel(S, R, n):
    spec = synthetic(S, R, 100 + R, init_mean=40.0, bounded=True)
    total = workloads.initial_total_propensity(spec)
    g = build_device(spec, 9)
    tmax = 50.0 / total if total else 1.0
    name, out, st = _run(g, n, tmax)
    assert name.split(":")[0] == "incremental"
    name, lds, st2 = _run(g, n, tmax, kernel=K.REBOP_KERNEL_LDS)
    assert name.split(":")[0] == "lds"
    assert bool((out == lds).all()) and (st.events, st.draws) == (st2.events, st2.draws)


def test_the_incremental_kernel_s_forms():
    S = 40
    g, _ = _expr_net(S, [("0.1 * X1", None, [1] + [0] * (S - 1))] * 70, [3] * S, 1)
    assert _run(g, 5)[0] == "incremental:expr"
    # propensities are kept where their LDS costs no waves, or a jump is longer
    # than the update list can say
    assert _run(build_device(synthetic(33, 65, 1, bounded=True), 1), 5)[0] == "incremental:stored"
    spec = synthetic(128, 512, 7)
    assert _run(build_device(spec, 1), 64, 1e-4)[0] == "incremental"
    far = [0] * 128
    far[5] = 300
    assert _run(build_device((128, spec[1] + [(0.5, [0] * 128, far)], spec[2]), 1), 64, 1e-4)[0] == "incremental:stored"


def test_networks_the_incremental_kernel_leaves_to_the_lds_kernel():
    third = [0] * 40
    third[2] = 3
    spec = synthetic(40, 80, 5, bounded=True)
    assert _run(build_device((40, spec[1] + [(1e-6, third, [0] * 40)], spec[2]), 1), 5)[0] in ("lds:int16", "lds:int32")
    capped = build_device(spec, 1)
    capped.set_draw_cap(1 << 30)
    assert _run(capped, 5)[0].startswith("lds:int")
    # a launch that fills the chip, of a small network
    assert _run(build_device(synthetic(40, 40, 5, bounded=True), 1), 262_144, 1e-3)[0].startswith("lds:int")
    x0 = [2**40] + [5] * 39
    assert _run(build_device((40, spec[1], x0), 1), 5, 1e-18)[0] == "lds:int64"


def test_a_rerun_names_both():
    S = 40
    rx = [(5.0, [0] * S, [2**20] + [0] * (S - 1))] + [(0.1, [0] * S, [0] * S)] * 70
    name, out, _ = _run(build_device((S, rx, [2**30 - 2**20] + [0] * (S - 1)), 1), 6, tmax=4.0)
    assert name in ("incremental > lds:int64", "incremental:stored > lds:int64")
    assert int(out.max()) > 2**30


def test_the_lanes_of_a_trajectory():
    s = sir()
    for n, nb, want in [(1, 7, "g16"), (4096, 7, "g16"), (4097, 7, "g4"), (16_385, 7, "g2"), (40_000, 7, "main+g4"),
                        (5, 2048, "g4_far"), (20_000, 2048, "g2_far")]:
        assert _run(build_device(s, 1), n, 1.0, nb)[0] == "specialized:" + want, n
    assert _run(build_device(s, 1), 40_000, 1.0, kernel=PERSISTENT | K.REBOP_KERNEL_WHOLE)[0] == "specialized:main"
    for flag, want in ((K.REBOP_KERNEL_GROUP4, "g4"), (K.REBOP_KERNEL_GROUP2, "g2"), (0, "main")):
        assert _run(build_device(s, 1), 9, 1.0, kernel=SPEC | flag)[0] == "specialized:" + want
    assert _run(build_device(synthetic(20, 33, 2, bounded=True), 1), 9)[0] == "specialized:g4"
    capped = build_device(s, 1)
    capped.set_draw_cap(1 << 30)
    assert _run(capped, 9, 1.0)[0] == "specialized:g4"
    assert _run(build_device(s, 1), 9, 1.0, kernel=K.REBOP_KERNEL_PLAIN)[0] == "register:plain"
    assert _run(build_device(s, 1), 9, 1.0, kernel=K.REBOP_KERNEL_PERSISTENT)[0] == "register:persistent"


def test_other_entry_points():
    import torch

    g = build_device(dimers(), 1)
    g.run_all_events(0.01, n_traj=5)
    assert K.last_kernel() == "specialized:ev4_write"
    counts = torch.zeros(20_000, dtype=torch.int64, device="cuda")
    g.run_all_events_device(0.001, 20_000, counts.data_ptr())
    assert K.last_kernel() == "specialized:ev2_count"
    b = g.batch(10)
    b.advance_until(0.01)
    assert K.last_kernel() == "specialized:g16"
    large = build_device(synthetic(40, 80, 5, bounded=True), 1)
    b = large.batch(3)
    b.advance_until(0.001)
    assert K.last_kernel() == "lds:int64"
    out = torch.zeros((3, 4, 6), dtype=torch.int64, device="cuda")
    rates = torch.ones((2, 5), dtype=torch.float64, device="cuda")
    g.run_sweep_device(2, 3, 0.01, 2, out.data_ptr(), rates_ptr=rates.data_ptr())
    assert K.last_kernel() == "specialized:sweep"
    spec = synthetic(12, 90, 3, bounded=True)
    net = build_device(spec, 3)
    buf = torch.zeros((3, 12, 9), dtype=torch.int64, device="cuda")
    run_jobs([dict(net=net, tmax=0.01, nb_steps=2, n_traj=9, traj_begin=0, out_ptr=buf.data_ptr())])
    torch.cuda.synchronize()
    assert K.last_kernel() == "incremental:stored"
    _, want, _, _, _ = build_oracle(spec, sparse=True).run_grid(3, spec[2], 0.01, 2, n_traj=9)
    assert np.array_equal(buf.cpu().numpy(), want)
