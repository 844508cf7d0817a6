"""Cotangents that are no plain tensors: a batch under torch.func.vmap and a
lazily negated view, on host and device tensors."""
import numpy as np
import pytest

from dgpr_amd import cases, dgx

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("where", ["cpu", "cuda"])
def test_batched_cotangent_of_the_energy(where):
    from dgpr_amd import torch_adjoint as ta
    c = cases.tgv_case(n=2, p=2, seed=3, M=0.3, Re=400.0)
    with dgx.Solver(c.mesh, c.params) as s:
        U = torch.tensor(c.U0, dtype=torch.float64, device=where, requires_grad=True)
        mu = torch.tensor(c.params.mu, dtype=torch.float64, device=where, requires_grad=True)
        J = ta.kinetic_energy_after_rk4(U, mu, s, c.dt, 2)
        ref = torch.autograd.grad(J, (U, mu), retain_graph=True)
        v = torch.tensor([1.0, -2.5, 0.0], dtype=torch.float64, device=where)
        got = torch.func.vmap(lambda x: torch.autograd.grad(J, (U, mu), x, retain_graph=True))(v)
        for g, r in zip(got, ref):
            assert torch.equal(g, v.view(-1, *[1] * r.dim()) * r)


def test_negated_view_as_cotangent():
    from dgpr_amd import torch_adjoint as ta
    c = cases.tgv_case(n=2, p=1, seed=4, M=0.3, Re=400.0)
    with dgx.Solver(c.mesh, c.params) as s:
        U = torch.tensor(c.U0, dtype=torch.float64, device="cuda", requires_grad=True)
        f = ta.residual(U, s)
        w = torch.tensor(np.random.default_rng(5).standard_normal(c.U0.size), device="cuda")
        (ref,) = torch.autograd.grad(f, U, w, retain_graph=True)
        (got,) = torch.autograd.grad(f, U, torch._neg_view(w))
        assert torch.equal(got, -ref)
