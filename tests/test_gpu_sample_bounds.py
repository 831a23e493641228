"""Where the grouped rounds store their samples.  A straight round also issues
stores for lanes and samples past the end, which the buffer's bounds check
drops: nothing around an output may change.  Offsets into the output are 32
bits wide, so an output near 4 GiB is compared on both sides of the line."""

from __future__ import annotations

import numpy as np
import pytest

from rebop_amd import _native as K
from tests.networks import build_device, build_oracle, dimers, sir

pytestmark = pytest.mark.gpu
SPEC = K.REBOP_KERNEL_PLAIN | K.REBOP_KERNEL_SPECIALIZED
PERSISTENT = K.REBOP_KERNEL_PERSISTENT | K.REBOP_KERNEL_SPECIALIZED


@pytest.mark.parametrize("kernel,n", [(K.REBOP_KERNEL_AUTO, 1), (K.REBOP_KERNEL_AUTO, 37), (K.REBOP_KERNEL_AUTO, 4096),
                                      (SPEC | K.REBOP_KERNEL_GROUP4, 37), (SPEC | K.REBOP_KERNEL_GROUP2, 37),
                                      (PERSISTENT, 70_001)])
@pytest.mark.parametrize("name,nb", [("sir", 1), ("sir", 6), ("decay", 31), ("dimers", 9)])
def test_nothing_around_the_samples_changes(name, nb, kernel, n, nthreads):
    import torch

    spec, tmax = {"sir": (sir(), 60.0), "dimers": (dimers(), 0.05),
                  "decay": ((2, [(1.0, [1, 0], [-1, 1])], [9, 0]), 3.0)}[name]
    size, guard = (nb + 1) * spec[0] * n, 32 * spec[0] * n  # a round stores up to 17 samples past the end
    buf = torch.full((guard + size + guard,), -7, dtype=torch.int64, device="cuda")
    out = buf[guard:guard + size]
    fin = torch.full((3 * spec[0] * n,), -7, dtype=torch.int64, device="cuda")
    g = build_device(spec, 23)
    g.run_device(tmax, nb, n, out.data_ptr(), final_ptr=fin[spec[0] * n:].data_ptr(), kernel=kernel, traj_begin=5)
    torch.cuda.synchronize()
    assert bool((buf[:guard] == -7).all()) and bool((buf[guard + size:] == -7).all())
    assert bool((fin[:spec[0] * n] == -7).all()) and bool((fin[2 * spec[0] * n:] == -7).all())
    _, oout, _, _, _ = build_oracle(spec).run_grid(23, spec[2], tmax, nb, n_traj=n, traj_begin=5, nthreads=nthreads)
    assert np.array_equal(out.view(nb + 1, spec[0], n).cpu().numpy(), oout)
    assert np.array_equal(fin[spec[0] * n:2 * spec[0] * n].view(spec[0], n).cpu().numpy(), oout[nb])


@pytest.mark.parametrize("kernel", [K.REBOP_KERNEL_AUTO, SPEC | K.REBOP_KERNEL_GROUP4, SPEC | K.REBOP_KERNEL_GROUP2])
def test_no_samples_at_all(kernel):
    """Final counts only: the straight rounds have no output to store to."""
    import torch

    g = build_device(sir(), 23)
    fin = torch.zeros((3, 41), dtype=torch.int64, device="cuda")
    g.run_device(60.0, 7, 41, None, final_ptr=fin.data_ptr(), kernel=kernel)
    torch.cuda.synchronize()
    _, oout, _, _, _ = build_oracle(sir()).run_grid(23, sir()[2], 60.0, 7, n_traj=41)
    assert np.array_equal(fin.cpu().numpy(), oout[7])


# 32 species x 8192 trajectories: 2 MiB a sample, with the 24 that a round may
# run past the end 2047 samples below 4 GiB (straight rounds), 2049 above
@pytest.mark.parametrize("samples", [2023, 2025])
@pytest.mark.parametrize("kernel", [K.REBOP_KERNEL_AUTO, SPEC | K.REBOP_KERNEL_GROUP2])
def test_outputs_around_4_gib(samples, kernel, nthreads):
    import torch

    S, n, nb = 32, 8192, samples - 1
    rx = []
    for a, b, k in ((0, 31, 0.4), (31, 17, 0.2), (17, 0, 0.3)):  # a cycle: never absorbed
        orders, d = [0] * S, [0] * S
        orders[a] = 1
        d[a], d[b] = -1, 1
        rx.append((k, orders, d))
    spec = (S, rx, [3 if s in (0, 17, 31) else s for s in range(S)])
    size, guard = samples * S * n, 32 * S * n
    buf = torch.full((size + guard,), -7, dtype=torch.int64, device="cuda")
    build_device(spec, 3).run_device(12.0, nb, n, buf.data_ptr(), kernel=kernel)
    other = torch.full((size,), -7, dtype=torch.int64, device="cuda")
    build_device(spec, 3).run_device(12.0, nb, n, other.data_ptr(), kernel=PERSISTENT | K.REBOP_KERNEL_WHOLE)
    torch.cuda.synchronize()
    assert bool((buf[size:] == -7).all())
    assert torch.equal(buf[:size], other)
    last = buf[:size].view(samples, S, n)[:, :, n - 3:].cpu().numpy()
    _, oout, _, _, _ = build_oracle(spec, sparse=True).run_grid(3, spec[2], 12.0, nb, n_traj=3, traj_begin=n - 3,
                                                                nthreads=nthreads)
    assert np.array_equal(last, oout)


def test_the_tail_of_an_output_beyond_4_gib(nthreads):
    """The last trajectories of a persistent run go to a grouped launch, whose
    offsets would not fit: 1.1e6 dimer trajectories x 127 samples, 4.5 GB."""
    import torch

    n, nb, tmax = 1_100_000, 126, 0.02
    out = torch.full(((nb + 1) * 4 * n + 4 * n,), -7, dtype=torch.int64, device="cuda")
    st = build_device(dimers(), 5).run_device(tmax, nb, n, out.data_ptr(), kernel=PERSISTENT)
    whole = torch.full(((nb + 1) * 4 * n,), -7, dtype=torch.int64, device="cuda")
    build_device(dimers(), 5).run_device(tmax, nb, n, whole.data_ptr(), kernel=PERSISTENT | K.REBOP_KERNEL_WHOLE)
    torch.cuda.synchronize()
    assert st.tail > 0
    assert torch.equal(out[:-4 * n], whole) and bool((out[-4 * n:] == -7).all())
    last = whole.view(nb + 1, 4, n)[:, :, n - 4:].cpu().numpy()
    _, oout, _, _, _ = build_oracle(dimers()).run_grid(5, dimers()[2], tmax, nb, n_traj=4, traj_begin=n - 4,
                                                       nthreads=nthreads)
    assert np.array_equal(last, oout)
