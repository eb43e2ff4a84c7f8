"""Functional calls whose output is one of their inputs: a residual with a general LDG beta
over its own state, and a VJP over its cotangent.  Meshes of more workgroups than run at once
on few elements per workgroup, so that a launch which still read its neighbours' states (or
cotangents) while it wrote would read some of them overwritten."""

from __future__ import annotations

import numpy as np
import pytest

from common import TWO_PI, paired, residual_parity

pytestmark = pytest.mark.gpu


def _case(n, order, viscous, extra):
    D = len(n)
    return dict(name=f"inpl_{'x'.join(map(str, n))}_p{order}_{viscous}_" + "_".join(map(str, extra.values())), n=n,
                lo=(0.0,) * D, hi=(TWO_PI,) * D, order=order, viscous=viscous, state="smooth", extra=extra)


@pytest.mark.parametrize("n,order,beta,flux", [((40, 41), 3, 0.2, "Rusanov"), ((12, 11, 13), 2, 0.0, "Roe"),
                                               ((7, 6, 8), 3, -0.3, "Rusanov"), ((3, 3, 4), 6, 0.2, "Rusanov")])
def test_general_beta_residual_over_its_state(n, order, beta, flux):
    z, o, _ = paired(_case(n, order, True, {"ldg_b": beta, "fconv_type": flux}))
    o.compute_residual(0)
    for tile in (0, 1):
        z.set_tile(tile)
        U = z.state_tensor()
        assert z.residual_at(U, U) is U
        got = U.cpu().numpy().transpose(2, 1, 0)
        err, kappa, ok = residual_parity(got, o)
        assert ok, f"tile {tile}: relative error {err:.2e}, condition {kappa:.1e}"


@pytest.mark.parametrize("n,order,viscous,extra", [
    ((40, 41), 2, False, {"fconv_type": "Roe"}), ((30, 31), 4, True, {"ldg_b": 0.5}),
    ((8, 7, 9), 3, True, {"ldg_b": -0.5, "fconv_type": "Roe"}), ((9, 8, 7), 2, True, {"ldg_b": 0.2})])
def test_vjp_over_its_cotangent(n, order, viscous, extra):
    import torch
    z, _, _ = paired(_case(n, order, viscous, extra))
    U = z.state_tensor()
    w = torch.randn(U.shape, dtype=torch.float64, generator=torch.Generator().manual_seed(5)).cuda()
    ref = z.residual_vjp(U, w)
    assert z.residual_vjp(U, w, w) is w
    np.testing.assert_array_equal(w.cpu().numpy(), ref.cpu().numpy())
