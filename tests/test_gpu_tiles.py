"""Launches at tiles of one to several elements per workgroup: what a workgroup of several
waves, a ragged last workgroup or elements of different numbers of face passes beside each
other could change, against one element per workgroup."""

from __future__ import annotations

import numpy as np
import pytest

from common import TWO_PI, paired

pytestmark = pytest.mark.gpu


def _solver(n, order, viscous, beta, flux):
    D = len(n)
    z, _, _ = paired(dict(name=f"tile_{'x'.join(map(str, n))}_p{order}_{viscous}_{beta}_{flux}", n=n, lo=(0.0,) * D,
                          hi=(TWO_PI,) * D, order=order, viscous=viscous, state="smooth",
                          extra={"ldg_b": beta, "fconv_type": flux}))
    return z


@pytest.mark.parametrize("n", [(11, 9, 10), (33, 32, 31), (34, 31, 32), (41, 40, 40)])
@pytest.mark.parametrize("viscous", [True, False])
def test_default_tile_of_one_point_elements(n, viscous):
    """990 (32 per workgroup), 32736 and 33728 (32 and 33) and 65600 hexes (64)."""
    z = _solver(n, 0, viscous, 0.5, "Rusanov")
    U = z.state_tensor()
    ref = z.residual_at(U).cpu().numpy()
    z.set_tile(1)
    np.testing.assert_array_equal(z.residual_at(U).cpu().numpy(), ref)
