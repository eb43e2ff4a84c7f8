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


def _close(got, ref):
    """Rounding apart (kernels of one wave and of several are separate compilations): per
    variable within 1e-12 of the largest entry, the bound of the residual's parity."""
    for v in range(ref.shape[1]):
        assert np.abs(got[:, v] - ref[:, v]).max() <= 1e-12 * np.abs(ref[:, v]).max(), v


@pytest.mark.parametrize("n,order", [((13, 3), 1), ((11, 5), 2), ((7, 5), 4), ((5, 5), 5), ((3, 3, 5), 1),
                                     ((3, 4, 5), 2), ((3, 3, 3), 3)])
@pytest.mark.parametrize("viscous,beta,flux", [(False, 0.5, "Rusanov"), (False, 0.5, "Roe"), (True, 0.5, "Rusanov"),
                                               (True, -0.5, "Roe"), (True, 0.2, "Rusanov"), (True, 0.0, "Roe")])
def test_every_tile_gives_the_same_vjp(n, order, viscous, beta, flux):
    import torch
    z = _solver(n, order, viscous, beta, flux)
    U = z.state_tensor()
    w = torch.randn(U.shape, dtype=torch.float64, generator=torch.Generator().manual_seed(11)).cuda()
    z.set_tile(1)
    ref = z.residual_vjp(U, w).cpu().numpy()
    assert np.isfinite(ref).all()
    for tile in (0, 2, 3, 64):  # 0: the default; 64: as many as fit
        z.set_tile(tile)
        _close(z.residual_vjp(U, w).cpu().numpy(), ref)


@pytest.mark.parametrize("n,order,beta,flux", [((7, 5), 4, 0.0, "Rusanov"), ((5, 3), 7, 0.2, "Roe"),
                                               ((13, 3), 1, -0.2, "Rusanov"), ((3, 4, 3), 2, 0.2, "Roe"),
                                               ((3, 3, 3), 3, 0.0, "Rusanov"), ((3, 3, 5), 1, 0.0, "Roe"),
                                               ((5, 4), 7, 0.5, "Rusanov"), ((4, 5), 7, -0.5, "Roe"),
                                               ((5, 3), 8, 0.5, "Rusanov"), ((3, 5), 8, -0.5, "Roe")])
def test_every_tile_gives_the_same_viscous_residual(n, order, beta, flux):
    from common import residual_parity
    D = len(n)
    z, o, _ = paired(dict(name=f"tiler_{'x'.join(map(str, n))}_p{order}_{beta}_{flux}", n=n, lo=(0.0,) * D,
                          hi=(TWO_PI,) * D, order=order, viscous=True, state="smooth",
                          extra={"ldg_b": beta, "fconv_type": flux}))
    o.compute_residual(0)
    ref = None
    for tile in (1, 0, 2, 3, 64):
        z.set_tile(tile)
        z.compute_residual(0)
        got = z.state("divF", 0)
        if ref is None:
            ref = got
            err, kappa, ok = residual_parity(got, o)
            assert ok, f"relative error {err:.2e}, condition {kappa:.1e}"
        _close(got, ref)


def test_no_residual_has_a_trace_launch():
    """Autotuned tiles of a general LDG beta: the first phase launches nothing, so its entry is
    the solver-wide tile, as in the other cases."""
    z = _solver((8, 8), 3, True, 0.2, "Rusanov")
    z.autotune(5)
    t = z.tiles()
    assert t[0] == t[1] and min(t) >= 1, t
