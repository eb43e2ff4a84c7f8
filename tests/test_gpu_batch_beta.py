"""Batches of general-beta members: a trace launch and the both-sides pair per order and element
type, against each member's own residual."""

from __future__ import annotations

import numpy as np
import pytest

from common import TWO_PI, paired

pytestmark = pytest.mark.gpu


def test_general_beta_members_of_a_batch():
    """Within 1e-14 of the largest entry (separate compilations of the same arithmetic, and
    traces read instead of extrapolated), over several replays."""
    from zefr_amd.zefr import Batch
    zs, refs = [], []
    for n, order, beta, flux in (((9, 8), 1, 0.2, "Rusanov"), ((5, 4), 1, 0.0, "Rusanov"), ((4, 5), 5, 0.0, "Roe"),
                                 ((3, 4), 8, 0.2, "Rusanov"), ((3, 3, 4), 1, -0.2, "Roe"),
                                 ((3, 3, 3), 3, 0.0, "Rusanov"), ((2, 3, 2), 6, 0.2, "Rusanov"),
                                 ((1, 2, 3), 2, 0.2, "Rusanov")):
        D = len(n)
        z, _, _ = paired(dict(name=f"bb_{'x'.join(map(str, n))}_p{order}_{beta}_{flux}", n=n, lo=(0.0,) * D,
                              hi=(TWO_PI,) * D, order=order, viscous=True, state="smooth",
                              extra={"ldg_b": beta, "fconv_type": flux}))
        z.compute_residual(0)
        refs.append(z.state("divF", 0, layout="device").copy())
        zs.append(z)
    b = Batch(zs)
    for _ in range(3):
        for z, r in zip(zs, refs):
            z._copy(2, 0, np.zeros_like(r), True)
        b.residual()
        for k, (z, r) in enumerate(zip(zs, refs)):
            got = z.state("divF", 0, layout="device")
            assert np.abs(got - r).max() <= 1e-14 * np.abs(r).max(), k
