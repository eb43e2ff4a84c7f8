"""The solution traces that launches read from Utr or write for the next one."""

from __future__ import annotations

import ctypes as C

import pytest

from ele_block import Block, ok, ptr
from zefr_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,order,first", [(2, 0, 3), (2, 1, 3), (3, 0, 5), (3, 1, 4), (3, 2, 6), (2, 4, 3), (3, 3, 3),
                                           (3, 6, 3)])
@pytest.mark.parametrize("beta,flux", [(0.5, 0), (-0.5, 2)])
def test_traced_gradient_flux_only_reads_the_trace(D, order, first, beta, flux):
    """The whole trace is as zfr_extrapolate left it, also at the points of elements that own
    more flux points than they have solution points, and the results are zfr_gradient_flux's."""
    import torch
    L, b = _lib.lib(), Block(D, order, first=first)
    for tile in (0, 3):
        d, out = b.desc(beta=beta, flux=flux, tile=tile), []
        for traced in (False, True):
            dF = b.field()
            b.Ftr.zero_()
            if traced:
                b.Utr.fill_(7.0)
                torch.cuda.synchronize()
                ok(L.zfr_extrapolate(C.byref(d), ptr(b.U), None))
                torch.cuda.synchronize()
                before = b.Utr.clone()
                torch.cuda.synchronize()
                ok(L.zfr_gradient_flux_traced(C.byref(d), ptr(b.U), ptr(dF), None))
                torch.cuda.synchronize()
                assert torch.equal(b.Utr, before)
            else:
                torch.cuda.synchronize()
                ok(L.zfr_gradient_flux(C.byref(d), ptr(b.U), ptr(dF), None))
                torch.cuda.synchronize()
            out.append((dF, b.Ftr.clone()))
        assert torch.isfinite(out[0][0]).all() and out[0][1].abs().sum() > 0
        assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])


@pytest.mark.parametrize("order", [5, 6, 7, 8])
@pytest.mark.parametrize("viscous,beta,flux", [(False, 0.5, "Rusanov"), (True, 0.5, "Roe"), (True, -0.5, "Rusanov"),
                                               (True, 0.2, "Rusanov")])
def test_fused_steps_of_large_hexes(order, viscous, beta, flux):
    """Steps whose stages hand traces on (hexes of order 6 to 8) or form them from the stage
    states (order 5), launched or replayed from a graph: U, U_ini and every stage's residual
    equal the plain sequence's."""
    import numpy as np
    from common import TWO_PI, paired
    n, z = (2, 3, 2), []
    for fuse, graph in ((False, False), (True, False), (True, True)):
        s, _, _ = paired(dict(name=f"hand_p{order}_{viscous}_{beta}_{flux}", n=n, lo=(0.0,) * 3, hi=(TWO_PI,) * 3,
                              order=order, viscous=viscous, state="smooth", extra={"ldg_b": beta, "fconv_type": flux}))
        s.set_step_mode(fuse, graph)
        for _ in range(3):
            s.do_step()
        z.append(s)
    for s in z[1:]:
        np.testing.assert_array_equal(s.state("U"), z[0].state("U"))
        np.testing.assert_array_equal(s.state("U_ini"), z[0].state("U_ini"))
        for stage in range(4):
            np.testing.assert_array_equal(s.state("divF", stage), z[0].state("divF", stage))


SHAPES = [(2, 0, 2), (2, 1, 3), (2, 4, 3), (2, 5, 2), (3, 1, 4), (3, 2, 3), (3, 3, 5), (3, 6, 3)]


def _stage(b, dF, X, tr):
    from test_cabi import _RkArgs
    return _RkArgs(U=ptr(X), U_ini=ptr(b.U), divF0=ptr(dF), mode=1, stage=0, nStages=4, alpha=0.5, dt=1e-3,
                   trace_out=ptr(tr))


@pytest.mark.parametrize("D,order,first", SHAPES)
@pytest.mark.parametrize("beta", [0.5, -0.5])
def test_face_correction_writes_the_next_trace(D, order, first, beta):
    """zfr_face_correction_rk with trace_out: the partner-owned half of the new state's trace,
    as zfr_extrapolate_partner writes it, the other points untouched; the next launch reads it."""
    import torch
    L, b = _lib.lib(), Block(D, order, first=first)
    owner = 0 if beta == 0.5 else 1
    for tile in (0, 1, 3, 4):
        d, dF, X = b.desc(beta=beta, tile=tile), b.field(), b.field()
        b.Utr.fill_(7.0)
        want, tr = b.Utr.clone(), b.Utr.clone()
        torch.cuda.synchronize()
        ok(L.zfr_gradient_flux(C.byref(d), ptr(b.U), ptr(dF), None))
        ok(L.zfr_face_correction_rk(C.byref(d), ptr(dF), C.byref(_stage(b, dF, X, tr)), None))
        d.Utr = ptr(want)
        ok(L.zfr_extrapolate_partner(C.byref(d), ptr(X), None))
        torch.cuda.synchronize()
        assert torch.isfinite(X).all() and not torch.equal(X, b.U)
        assert torch.equal(tr, want)
        assert torch.equal((tr == 7.0).all(1), b.slot == owner)
        R = [b.field(), b.field()]
        torch.cuda.synchronize()
        d.Utr = ptr(tr)
        ok(L.zfr_gradient_flux_traced(C.byref(d), ptr(X), ptr(R[0]), None))
        ok(L.zfr_face_correction(C.byref(d), ptr(R[0]), None))
        d.Utr = ptr(b.Utr)
        ok(L.zfr_gradient_flux(C.byref(d), ptr(X), ptr(R[1]), None))
        ok(L.zfr_face_correction(C.byref(d), ptr(R[1]), None))
        torch.cuda.synchronize()
        assert torch.equal(R[0], R[1])


@pytest.mark.parametrize("D,order,first", SHAPES)
@pytest.mark.parametrize("beta", [0.2, 0.0])
def test_both_sides_correction_writes_the_next_trace(D, order, first, beta):
    """zfr_both_sides_correction with trace_out: the whole trace, as zfr_extrapolate writes it
    (which zfr_gradient and zfr_divergence read)."""
    import torch
    L, b = _lib.lib(), Block(D, order, first=first)
    for tile in (0, 1, 3, 4):
        d, dF, X = b.desc(beta=beta, tile=tile), b.field(), b.field()
        tr = torch.full_like(b.Utr, 7.0)
        b.Utr.fill_(7.0)
        torch.cuda.synchronize()
        ok(L.zfr_both_sides_flux(C.byref(d), ptr(b.U), ptr(dF), None))
        ok(L.zfr_both_sides_correction(C.byref(d), ptr(dF), C.byref(_stage(b, dF, X, tr)), None))
        ok(L.zfr_extrapolate(C.byref(d), ptr(X), None))
        torch.cuda.synchronize()
        assert torch.isfinite(X).all() and not torch.equal(X, b.U)
        assert torch.equal(tr, b.Utr)
