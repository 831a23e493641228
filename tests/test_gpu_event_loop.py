"""GPU parity of the specialised kernels' event loop at the edges of its
shortcuts, against the CPU oracle, bit for bit: totals outside the range of
the plain division, and jumps read as fields of one word."""

from __future__ import annotations

import numpy as np
import pytest

from rebop_amd import _native as K
from tests.networks import build_device, build_oracle

pytestmark = pytest.mark.gpu
SPEC = K.REBOP_KERNEL_SPECIALIZED
KINDS = [K.REBOP_KERNEL_PERSISTENT | SPEC, K.REBOP_KERNEL_PLAIN | SPEC | K.REBOP_KERNEL_GROUP2,
         K.REBOP_KERNEL_PLAIN | SPEC | K.REBOP_KERNEL_GROUP4, K.REBOP_KERNEL_PERSISTENT]


def _same(spec, tmax, nb, n, kernel, nthreads, seed=19):
    import torch

    g = build_device(spec, seed)
    out = torch.zeros((nb + 1, spec[0], n), dtype=torch.int64, device="cuda")
    st = g.run_device(tmax, nb, n, out.data_ptr(), kernel=kernel, traj_begin=2)
    torch.cuda.synchronize()
    _, oout, _, oev, odr = build_oracle(spec).run_grid(seed, spec[2], tmax, nb, n_traj=n, traj_begin=2,
                                                       nthreads=nthreads)
    assert np.array_equal(out.cpu().numpy(), oout)
    assert (st.events, st.draws) == (oev, odr)
    return oout, oev


# 2^-700 = 1.9e-211 and 2^700 = 5.3e210 bound the plain division; the totals
# of sixty decaying particles cross them for two of these constants
@pytest.mark.parametrize("k", [1e-290, 5e-309, 4e-213, 8e209, 1e290])
@pytest.mark.parametrize("kernel", KINDS)
def test_totals_far_from_one(k, kernel, nthreads):
    spec = (2, [(k, [1, 0], [-1, 1])], [60, 0])
    oout, oev = _same(spec, 3.0 / k if k > 1e-300 else 1e308, 13, 70, kernel, nthreads)
    assert oev > 70


# the largest difference sets the field's width, and (reactions + 1) fields
# have to fit 32 bits: 2 bits up to 15 reactions, 4 up to 7, 8 up to 3, 16: 1
@pytest.mark.parametrize("R,jump", [(15, 1), (16, 1), (7, 3), (7, -8), (7, 8), (8, 7), (3, 127), (3, 128), (4, 100),
                                    (3, -128)])
@pytest.mark.parametrize("kernel", KINDS[:3])
def test_jumps_as_fields_of_a_word(R, jump, kernel, nthreads):
    S = 3
    up = abs(jump)
    rx = [(2.0, [0, 0, 0], [up, 0, 0])] if jump > 0 else [(1e-3, [up, 0, 0] if up <= 8 else [1, 0, 0], [jump, 1, 0])]
    for r in range(1, R):
        a = r % S
        o, d = [0] * S, [0] * S
        o[a] = 1
        d[a], d[(a + 1) % S] = -1, 1
        rx.append((0.05 * r, o, d))
    _same((S, rx, [200, 40, 30]), 2.0, 9, 70, kernel, nthreads)
