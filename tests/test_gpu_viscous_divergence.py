"""The three viscous launches zfr_extrapolate, zfr_gradient and zfr_divergence (also with an
update) against the two-launch residuals: one flux, formed on both sides of a face there and
handed across it here."""

from __future__ import annotations

import ctypes as C

import pytest

from ele_block import Block, ok, ptr
from test_cabi import _RkArgs
from zefr_amd import _lib

pytestmark = pytest.mark.gpu


def _close(got, ref):
    """Per variable within 1e-12 of the largest entry, the bound of the residual's parity: sums
    of some ten terms of the results' own size, in another order."""
    import torch
    assert torch.isfinite(ref).all()
    for v in range(ref.shape[1]):
        assert (got[:, v] - ref[:, v]).abs().max() <= 1e-12 * ref[:, v].abs().max(), v


@pytest.mark.parametrize("D,order,first", [(2, 0, 2), (2, 1, 3), (2, 4, 3), (3, 1, 4), (3, 2, 3), (3, 3, 5), (3, 6, 3)])
@pytest.mark.parametrize("beta", [0.5, -0.5, 0.2, 0.0])
@pytest.mark.parametrize("flux", [0, 2])
def test_three_launches_give_the_two_launch_residual(D, order, first, beta, flux):
    import torch
    L, b = _lib.lib(), Block(D, order, first=first)
    for tile in (0, 3):
        d, ref, dF, X = b.desc(beta=beta, flux=flux, tile=tile), b.field(), b.field(), [b.field(), b.field()]
        a = [_RkArgs(U=ptr(x), U_ini=ptr(b.U), mode=1, stage=0, nStages=4, alpha=0.5, dt=1e-3) for x in X]
        torch.cuda.synchronize()
        if beta in (0.5, -0.5):
            ok(L.zfr_gradient_flux(C.byref(d), ptr(b.U), ptr(ref), None))
            ok(L.zfr_face_correction_rk(C.byref(d), ptr(ref), C.byref(a[0]), None))
        else:
            ok(L.zfr_both_sides_flux(C.byref(d), ptr(b.U), ptr(ref), None))
            ok(L.zfr_both_sides_correction(C.byref(d), ptr(ref), C.byref(a[0]), None))
        ok(L.zfr_extrapolate(C.byref(d), ptr(b.U), None))
        ok(L.zfr_gradient(C.byref(d), ptr(b.U), None, None))
        ok(L.zfr_divergence(C.byref(d), ptr(b.U), ptr(dF), None))
        torch.cuda.synchronize()
        _close(dF, ref)
        ok(L.zfr_divergence_rk(C.byref(d), ptr(b.U), ptr(dF), C.byref(a[1]), None))
        torch.cuda.synchronize()
        _close(dF, ref)
        _close(X[1], X[0])
