"""A device element block with made-up geometry for kernel-level tests: elements 2k and 2k + 1
are partners at every flux point, and `first` of an even element's faces have slot 0 on its
side, so that elements may own most of their faces or few of them."""

from __future__ import annotations

import ctypes as C

import torch

from zefr_amd import _lib


def ptr(t):
    return C.c_void_p(t.data_ptr())


def ok(rc):
    assert rc == 0, _lib.last_error()


def zeros(*s):
    return torch.zeros(s, dtype=torch.float64, device="cuda")


class Block:
    def __init__(self, D, order, E=14, first=None, seed=3):
        N, V = order + 1, D + 2
        nS, nF = N ** D, 2 * D * N ** (D - 1)
        self.D, self.order, self.E, self.V, self.nS, self.nF = D, order, E, V, nS, nF
        g = torch.Generator().manual_seed(seed)
        r = lambda *s: torch.rand(s, generator=g, dtype=torch.float64)  # noqa: E731
        vel, rho, p = 0.3 * (r(E, D, nS) - 0.5), 1.0 + 0.1 * r(E, nS), 1.0 + 0.1 * r(E, nS)
        self.U = torch.cat([rho[:, None], rho[:, None] * vel, (p / 0.4 + 0.5 * rho * (vel ** 2).sum(1))[:, None]],
                           1).cuda()
        metric = 0.1 * r(E, D * D + 1, nS)
        for d in range(D):
            metric[:, d * D + d] += 1.0
        metric[:, D * D] += 1.0
        nrm = r(E // 2, D, nF) - 0.5
        nrm = (nrm / nrm.norm(dim=1, keepdim=True)).repeat_interleave(2, 0)  # slot 0's normal, on both sides
        e, f = torch.arange(E)[:, None], torch.arange(nF)[None]
        slot = (e & 1) ^ (f // N ** (D - 1) >= (D if first is None else first)).to(torch.int64)
        dA = (1.0 + r(E, nF)) * (1 - 2 * slot)
        bits = 8 if nF <= 256 else 9
        self.slot = slot.cuda()
        self.nbr = ((e ^ 1) << (bits + 1) | slot << bits | f).to(torch.int32).cuda()
        self.metric, self.fgeo = metric.cuda(), torch.cat([nrm, dA[:, None]], 1).contiguous().cuda()
        lE = r(2, N) + 0.1  # convex weights, so that every trace is a state with rho, p > 0
        self.ops = torch.cat([(lE / lE.sum(1, keepdim=True)).flatten(), r(N * N + 2 * N) - 0.5]).cuda()
        self.Utr, self.Gtr, self.Ftr = zeros(E, V, nF), zeros(E, D, V, nF), zeros(E, V, nF)

    def desc(self, viscous=1, beta=0.5, flux=0, tile=0):
        return _lib.EleDesc(nDims=self.D, order=self.order, nVars=self.V, nEles=self.E, nSpts=self.nS,
                            nFpts=self.nF, viscous=viscous, gamma=1.4, prandtl=0.72, mu=0.01, fix_vis=1, ldg_b=beta,
                            ldg_tau=0.1, fconv_type=flux, eles_per_block=tile, ops1d=ptr(self.ops),
                            metric=ptr(self.metric), fgeo=ptr(self.fgeo), nbr=ptr(self.nbr), Utr=ptr(self.Utr),
                            Gtr=ptr(self.Gtr), Ftr=ptr(self.Ftr))

    def field(self):
        return zeros(self.E, self.V, self.nS)
