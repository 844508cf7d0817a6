"""The device-pointer adjoint calls and the workspace that the adjoint calls
keep on the context: bit for bit the host forms', whatever call used the
workspace before, with and without dJ/dmu, and after a release."""
import numpy as np
import pytest

from dgpr_amd import cases, dgx

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p", [1, 2, 3])
def test_device_forms_equal_host_forms(p):
    c = cases.channel_case(3, 2, 3, p=p, seed=70 + p, nsteps=2)
    w = np.random.default_rng(p).standard_normal(c.U0.shape)
    with dgx.Solver(c.mesh, c.params) as s:
        def host():
            s.set_state(c.U0)
            g = s.residual_vjp(w)
            s.set_state(c.U0)
            J, gU, dmu = s.adjoint_rk4(c.dt, 3)
            return g, gU, J, dmu

        def device():
            wd = torch.tensor(w, device="cuda")
            g, gU = torch.empty_like(wd), torch.empty_like(wd)
            torch.cuda.synchronize()
            s.set_state(c.U0)
            J, dmu = s.adjoint_rk4_device(c.dt, 3, gU.data_ptr())
            s.set_state(c.U0)
            s.residual_vjp_device(wd.data_ptr(), g.data_ptr())
            return g.cpu().numpy(), gU.cpu().numpy(), J, dmu

        ref = host()
        runs = [device(), host()]
        s.adjoint_release()
        runs += [device()]
        s.adjoint_release()
        s.set_state(c.U0)
        _, gU, none = s.adjoint_rk4(c.dt, 3, want_mu=False)  # smaller workspace, then grown
        assert none is None and np.array_equal(gU, ref[1])
        runs += [host(), device()]
        for r in runs:
            assert all(np.array_equal(a, b) for a, b in zip(r, ref))
