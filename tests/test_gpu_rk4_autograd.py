"""The differentiated RK44 step as fused stage kernels (autograd.RK4Step) against the tensor
expressions it stands for, which rk4_step still takes for every call the kernels do not
cover (here: a numpy dt)."""

import numpy as np
import pytest

from common import TWO_PI, make_mesh, product, tmp, write_deck

pytestmark = pytest.mark.gpu

# elements per workgroup of the grid, points that do not fill a wave, both dimensions
CASES = [((3, 3), 1, True), ((5, 4), 4, False), ((3, 4, 3), 2, True), ((3, 3, 3), 3, False)]


def solver(n, order, viscous):
    D = len(n)
    name = "rk4ad_" + "x".join(map(str, n)) + f"_p{order}"
    mesh = make_mesh(name + ".msh", n, (0.0,) * D, (TWO_PI,) * D, 0.03)
    return product(write_deck(tmp(name + ".deck"), mesh, D, order, viscous))


def field(z, seed):
    import torch
    d = z.dims()
    g = torch.Generator().manual_seed(seed)
    r = lambda: torch.rand((d["nEles"], d["nSpts"]), generator=g, dtype=torch.float64) - 0.5  # noqa: E731
    rho, p, vel = 1.0 + 0.1 * r(), 1.0 + 0.1 * r(), [0.3 * r() for _ in range(d["nDims"])]
    E = p / 0.4 + 0.5 * rho * sum(v * v for v in vel)
    return torch.stack([rho] + [rho * v for v in vel] + [E], dim=1).cuda()


@pytest.mark.parametrize("n,order,viscous", CASES)
def test_fused_step_matches_tensor_expressions(n, order, viscous):
    import torch
    from zefr_amd.autograd import RK4Step, device_field, rk4_step
    z = solver(n, order, viscous)
    detJ = device_field(z, "jaco_det_spts")
    U0, c, dt = field(z, 1), torch.randn_like(field(z, 2)), 1e-3
    got = []
    for step in (dt, np.float64(dt)):  # fused, then the tensor expressions
        U = U0.clone().requires_grad_()
        Y = rk4_step(z, U, step, detJ)
        assert isinstance(Y.grad_fn, RK4Step._backward_cls) == (step is dt)
        got.append((Y.detach(), torch.autograd.grad((c * Y).sum(), U)[0]))
    (Ya, ga), (Yb, gb) = got
    eps = np.finfo(np.float64).eps
    # a few roundings per stage, of the size of the terms summed
    assert (Ya - Yb).abs().max() <= 8 * eps * Yb.abs().max()
    # the same, carried through four linear VJPs whose terms are at most of the gradient's size
    assert (ga - gb).abs().max() <= 64 * eps * max(gb.abs().max(), c.abs().max())


def test_fused_step_inputs_and_higher_order():
    """A non-contiguous state, a detJ that is not the solver's, two steps, and create_graph
    (the gradient's dependence on the incoming one is the identity in both forms)."""
    import torch
    from zefr_amd.autograd import checkpointed_rollout, device_field, rk4_step, rollout
    z = solver((4, 3), 2, True)
    detJ = 2.0 * device_field(z, "jaco_det_spts")
    d = z.dims()
    U0 = field(z, 3)
    Ut = torch.empty((d["nSpts"], d["nVars"], d["nEles"]), dtype=torch.float64, device="cuda").permute(2, 1, 0)
    Ut.copy_(U0)
    assert not Ut.is_contiguous()
    assert torch.equal(rk4_step(z, Ut, 1e-3, detJ), rk4_step(z, U0, 1e-3, detJ))
    second = []
    for dt in (1e-3, np.float64(1e-3)):
        U = U0.clone().requires_grad_()
        (g,) = torch.autograd.grad((rk4_step(z, U, dt, detJ) ** 3).sum(), U, create_graph=True)
        second.append(torch.autograd.grad(g.sum(), U)[0])
    assert torch.allclose(second[0], second[1], rtol=1e-12, atol=1e-12)
    U = U0.clone().requires_grad_()
    a = torch.autograd.grad((rollout(z, U, 1e-3, 3, detJ) ** 2).sum(), U)[0]
    b = torch.autograd.grad((checkpointed_rollout(z, U, 1e-3, 3, every=2, detJ=detJ) ** 2).sum(), U)[0]
    assert torch.equal(a, b)


def test_general_path_kept():
    """Calls the fused step does not cover keep the tensor expressions: detJ that is
    differentiated or broadcast, a tensor dt."""
    import torch
    from zefr_amd.autograd import RK4Step, device_field, rk4_step
    z = solver((3, 3), 2, False)
    detJ = device_field(z, "jaco_det_spts")
    U = field(z, 4).requires_grad_()
    dj = detJ.clone().requires_grad_()
    for step, j in ((1e-3, dj), (1e-3, detJ.expand_as(U)), (torch.tensor(1e-3, dtype=torch.float64), detJ)):
        Y = rk4_step(z, U, step, j)
        assert not isinstance(Y.grad_fn, RK4Step._backward_cls)
        assert torch.isfinite(torch.autograd.grad(Y.sum(), U)[0]).all()
    assert torch.isfinite(torch.autograd.grad(rk4_step(z, U, 1e-3, dj).sum(), dj)[0]).all()


def test_saved_tensor_hooks_and_dual_detJ():
    """Saved tensors that hooks hand back in another layout give the same gradient, one that comes
    back on the host is refused, and a detJ with a tangent takes the tensor expressions."""
    import torch
    from torch.autograd import forward_ad, graph
    from zefr_amd.autograd import RK4Step, _fusable, device_field, rk4_step
    z = solver((4, 3), 2, True)
    detJ, U0 = device_field(z, "jaco_det_spts"), field(z, 1)
    grads = []
    for hooks in (None, (lambda x: x, lambda x: x.transpose(0, -1).contiguous().transpose(0, -1))):
        U = U0.clone().requires_grad_()
        if hooks:
            with graph.saved_tensors_hooks(*hooks):
                Y = rk4_step(z, U, 1e-3, detJ)
        else:
            Y = rk4_step(z, U, 1e-3, detJ)
        assert isinstance(Y.grad_fn, RK4Step._backward_cls)
        grads.append(torch.autograd.grad(Y.square().sum(), U)[0])
    assert torch.equal(*grads)
    U = U0.clone().requires_grad_()
    with graph.saved_tensors_hooks(lambda x: x, lambda x: x.cpu() if x.shape == detJ.shape else x):
        Y = rk4_step(z, U, 1e-3, detJ)
    with pytest.raises(RuntimeError, match="detJ"):
        torch.autograd.grad(Y.sum(), U)
    with forward_ad.dual_level():
        assert _fusable(z, U0, 1e-3, detJ, None)
        assert not _fusable(z, U0, 1e-3, forward_ad.make_dual(detJ, torch.ones_like(detJ)), None)
