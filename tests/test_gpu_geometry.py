"""Geometry that a context lays out once: affine element records at the
general orders (unequal elements, several elements per workgroup, a partly
filled last one) and the stored geometry of q > 1 meshes, against the oracle
at the parity bars (f 1e-12, state 1e-10); Mach 0.2, where the rounding floor
of f is below 5e-13."""
import numpy as np
import pytest

from dgpr_amd import cases, dgx
from test_gpu_parity import DEFAULT_BOUNDS, RES_TOL, SOL_TOL, orc_params, rel
from test_gpu_tile import stretched_case

pytestmark = pytest.mark.gpu

CASES = {
    "p0_stretched_5x3x5": lambda: stretched_case(0, (5, 3, 5), [dgx.PERIODIC] * 6, 21),
    "p4_stretched_walls_2x1x2": lambda: stretched_case(4, (2, 1, 2), DEFAULT_BOUNDS, 22),
    "p5_stretched_1x2x1": lambda: stretched_case(5, (1, 2, 1), [dgx.PERIODIC] * 6, 23),
    "p1_q2_channel_3x2x3": lambda: cases.channel_case(3, 2, 3, p=1, q=2, seed=24, nsteps=3),
    "p1_q3_channel_3x1x1": lambda: cases.channel_case(3, 1, 1, p=1, q=3, seed=25, nsteps=3),
    "p2_q3_channel_1x3x1": lambda: cases.channel_case(1, 3, 1, p=2, q=3, seed=26, nsteps=3),
    "p1_q5_channel_3x3x1": lambda: cases.channel_case(3, 3, 1, p=1, q=5, seed=27, nsteps=3),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_against_oracle(name, orc):
    c = CASES[name]()
    m = c.mesh
    geo = orc.Geometry(m.p, m.q, m.nx, m.ny, m.nz, m.bounds, m.nodes)
    prm = orc_params(orc, c.params)
    R_o, f_o = geo.residual(prm, c.U0)
    U_o, n_o = geo.step(prm, c.U0, c.dt, c.scheme, 3)
    with dgx.Solver(m, c.params) as s:
        s.set_state(c.U0)
        R, f = s.residual()
        n = s.step(c.dt, c.scheme, 3)
        U = s.get_state()
    e = rel(f, f_o), rel(R, R_o), rel(U, U_o), float(np.max(np.abs(n / n_o - 1.0)))
    print(name, "f %.2e R %.2e state %.2e norms %.2e" % e, flush=True)
    assert e[0] < RES_TOL and e[1] < RES_TOL and e[2] < SOL_TOL and e[3] < SOL_TOL
