"""Fused RK steps whose stages extrapolate their partners' traces from the stage states, and
the kernel-level form that hands traces from stage to stage instead: the same numbers."""

from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from common import TWO_PI, paired
from test_cabi import _RkArgs
from zefr_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,order,flux", [((3, 4, 3), 1, "Rusanov"), ((3, 3, 4), 2, "Roe"), ((3, 3, 3), 3, "Rusanov"),
                                          ((5, 4), 0, "Rusanov"), ((4, 5), 4, "Roe")])
def test_euler_step_on_alternating_buffers(n, order, flux):
    """No stage writes the buffer it reads: U, U_ini and every stage's residual equal the plain
    sequence's bit for bit, also at a tile that leaves the last workgroup ragged."""
    D = len(n)
    z = []
    for fuse, tile in ((False, 0), (True, 0), (True, 2)):
        s, _, _ = paired(dict(name=f"stg{D}d_p{order}_{flux}", n=n, lo=(0.0,) * D, hi=(TWO_PI,) * D, order=order,
                              viscous=False, state="smooth", extra={"fconv_type": flux}))
        s.set_step_mode(fuse, False)
        if tile:
            s.set_tile(tile)
        for _ in range(3):
            s.do_step()
        z.append(s)
    for s in z[1:]:
        np.testing.assert_array_equal(s.state("U"), z[0].state("U"))
        np.testing.assert_array_equal(s.state("U_ini"), z[0].state("U_ini"))
        for stage in range(4):
            np.testing.assert_array_equal(s.state("divF", stage), z[0].state("divF", stage))


@pytest.mark.parametrize("D,order", [(3, 1), (3, 3), (2, 4)])
def test_trace_handed_to_the_next_stage(D, order):
    """zfr_gradient_flux_traced and an in-place zfr_divergence_rk read the trace a fused update
    (or zfr_extrapolate*) wrote; zfr_gradient_flux and a zfr_divergence_rk that writes another
    buffer form it from U.  Elements 2k and 2k + 1 are partners at every flux point."""
    import torch
    L, N, V, E = _lib.lib(), order + 1, D + 2, 14
    nS, nF = N ** D, 2 * D * N ** (D - 1)
    g = torch.Generator().manual_seed(3)
    r = lambda *s: torch.rand(s, generator=g, dtype=torch.float64)  # noqa: E731
    vel, rho, p = 0.3 * (r(E, D, nS) - 0.5), 1.0 + 0.1 * r(E, nS), 1.0 + 0.1 * r(E, nS)
    U = torch.cat([rho[:, None], rho[:, None] * vel, (p / 0.4 + 0.5 * rho * (vel ** 2).sum(1))[:, None]], 1).cuda()
    metric = (0.1 * r(E, D * D + 1, nS))
    for d in range(D):
        metric[:, d * D + d] += 1.0
    metric[:, D * D] += 1.0
    nrm = r(E // 2, D, nF) - 0.5
    nrm = (nrm / nrm.norm(dim=1, keepdim=True)).repeat_interleave(2, 0)  # slot 0's normal, on both sides
    e, f = torch.arange(E)[:, None], torch.arange(nF)[None]
    slot = (e & 1) ^ (f // N ** (D - 1) & 1)
    dA = (1.0 + r(E, nF)) * (1 - 2 * slot)
    nbr = ((e ^ 1) << 9 | slot << 8 | f).to(torch.int32).cuda()
    metric, fgeo = metric.cuda(), torch.cat([nrm, dA[:, None]], 1).contiguous().cuda()
    ops, z = r(N * N + 4 * N).cuda(), lambda *s: torch.zeros(s, dtype=torch.float64, device="cuda")  # noqa: E731
    Utr, Ftr = z(E, V, nF), z(E, V, nF)
    P = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731

    def desc(viscous):
        return _lib.EleDesc(nDims=D, order=order, nVars=V, nEles=E, nSpts=nS, nFpts=nF, viscous=viscous, gamma=1.4,
                            prandtl=0.72, mu=0.01, fix_vis=1, ldg_b=0.5, ldg_tau=0.1, ops1d=P(ops), metric=P(metric),
                            fgeo=P(fgeo), nbr=P(nbr), Utr=P(Utr), Ftr=P(Ftr))

    def ok(rc):
        assert rc == 0, _lib.last_error()
    d, out = desc(1), []
    for traced in (False, True):
        dF = z(E, V, nS)
        torch.cuda.synchronize()
        if traced:
            ok(L.zfr_extrapolate_partner(C.byref(d), P(U), None))
            ok(L.zfr_gradient_flux_traced(C.byref(d), P(U), P(dF), None))
        else:
            ok(L.zfr_gradient_flux(C.byref(d), P(U), P(dF), None))
        ok(L.zfr_face_correction(C.byref(d), P(dF), None))
        torch.cuda.synchronize()
        out.append(dF)
    assert torch.isfinite(out[0]).all() and torch.equal(out[0], out[1])
    # Euler, two stage updates: in place with the trace handed on, and between two buffers
    d, out = desc(0), []
    for in_place in (True, False):
        X, Y, dF, tr = U.clone(), z(E, V, nS), z(2, E, V, nS), z(E, V, nF)
        torch.cuda.synchronize()
        if in_place:
            ok(L.zfr_extrapolate(C.byref(d), P(X), None))
        for s, (src, dst) in enumerate(((X, X), (X, X)) if in_place else ((X, Y), (Y, X))):
            a = _RkArgs(U=P(dst), U_ini=P(U), mode=1, stage=s, nStages=4, alpha=0.5, dt=1e-3,
                        trace_out=P(tr) if in_place and s == 0 else None)
            if in_place:
                d.Utr = P(Utr) if s == 0 else P(tr)
            ok(L.zfr_divergence_rk(C.byref(d), P(src), P(dF[s]), C.byref(a), None))
        torch.cuda.synchronize()
        out.append((X, dF))
    assert torch.isfinite(out[0][0]).all() and not torch.equal(out[0][0], U)
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])
