"""Viscous residuals at tiles of one to several elements per workgroup: quads of five and more
points per direction deal the owned flux points of all the workgroup's elements to its threads
in a row, so elements that own more or fewer faces than half and a ragged last workgroup must
give what one element per workgroup gives, bit for bit, and match the oracle."""

from __future__ import annotations

import numpy as np
import pytest

from common import TWO_PI, paired, residual_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,order,beta,flux", [((13, 3), 4, 0.5, "Rusanov"), ((13, 3), 4, -0.5, "Roe"),
                                               ((7, 5), 5, -0.5, "Rusanov"), ((5, 4), 6, 0.5, "Roe"),
                                               ((3, 3), 9, 0.5, "Rusanov"), ((7, 3), 3, 0.5, "Rusanov"),
                                               ((7, 3), 1, -0.5, "Rusanov"), ((3, 4, 3), 2, 0.5, "Roe"),
                                               ((3, 3, 5), 1, 0.5, "Rusanov")])
def test_every_tile_gives_the_same_residual(n, order, beta, flux):
    D = len(n)
    z, o, _ = paired(dict(name=f"fi_{'x'.join(map(str, n))}_p{order}_{flux}_{beta}", n=n, lo=(0.0,) * D,
                          hi=(TWO_PI,) * D, order=order, viscous=True, state="smooth",
                          extra={"ldg_b": beta, "fconv_type": flux}))
    o.compute_residual(0)
    ref = None
    for tile in (1, 0, 2, 3, 64):  # 0: the default; 64: as many as fit
        z.set_tile(tile)
        z.compute_residual(0)
        got = z.state("divF", 0)
        if ref is None:
            ref = got
            err, kappa, ok = residual_parity(got, o)
            assert ok, f"relative error {err:.2e}, condition {kappa:.1e}"
        np.testing.assert_array_equal(got, ref)
