"""The tiled stage kernel where its inputs differ from the one-row kernel's:
it reads the neighbours' states and geometry instead of trace records, and of
the stored records only the boundary states of domain-boundary faces.

Meshes: element counts that leave a partly filled last tile, affine elements
of unequal size (the neighbour's J^-1 is not the own one), walls, inflow and
outflow.  Bars: the two kernels evaluate the same sums in another order, so f
agrees to a few hundred roundings of its largest terms (1e-12 relative at Mach
0.2 and above), the state after three steps to dt f of that (1e-13) and the
norms to 1e-12.
"""
import numpy as np
import pytest

from dgpr_amd import cases, dgx
from test_gpu_parity import DEFAULT_BOUNDS, perturbed_uniform, rel

pytestmark = pytest.mark.gpu


def stretched_case(p, nxyz, bounds, seed):
    """Affine box whose element sizes vary by a factor of about two."""
    rng = np.random.default_rng(seed)
    ax = []
    for n in nxyz:
        h = rng.uniform(0.7, 1.4, n)
        ax.append(np.concatenate([[0.0], np.cumsum(h / h.sum() * 2.0)]))
    nx, ny, nz = nxyz
    nodes = np.empty((nz, ny, nx, 2, 2, 2, 3))
    for c in range(2):
        nodes[:, :, :, :, :, c, 0] = ax[0][c:nx + c][None, None, :, None, None]
        nodes[:, :, :, :, c, :, 1] = ax[1][c:ny + c][None, :, None, None, None]
        nodes[:, :, :, c, :, :, 2] = ax[2][c:nz + c][:, None, None, None, None]
    mesh = dgx.Mesh(p, 1, nx, ny, nz, bounds, nodes)
    assert mesh.affine
    prm = dgx.make_reference_state(mu=5e-3, c=1.0, u=0.2)
    return cases.Case("stretched", mesh, prm, perturbed_uniform(mesh, prm, 0.03, seed), "RK4",
                      2e-3, 3)


def channel(p, nxyz, seed):
    return cases.channel_case(*nxyz, p=p, seed=seed, nsteps=3)


CASES = {
    "p1_stretched_5x3x1": lambda: stretched_case(1, (5, 3, 1), [dgx.PERIODIC] * 6, 1),
    "p1_stretched_walls_3x3x3": lambda: stretched_case(1, (3, 3, 3), DEFAULT_BOUNDS, 2),
    "p1_channel_3x3x3": lambda: channel(1, (3, 3, 3), 3),
    "p2_stretched_walls_5x1x3": lambda: stretched_case(2, (5, 1, 3), DEFAULT_BOUNDS, 4),
    "p2_channel_3x3x1": lambda: channel(2, (3, 3, 1), 5),
    "p3_stretched_3x3x3": lambda: stretched_case(3, (3, 3, 3), [dgx.PERIODIC] * 6, 6),
    "p3_stretched_walls_1x3x1": lambda: stretched_case(3, (1, 3, 1), DEFAULT_BOUNDS, 7),
    "p3_channel_3x1x3": lambda: channel(3, (3, 1, 3), 8),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_tiled_against_one_row(name):
    c = CASES[name]()
    got = {}
    for tile in (0, 1):
        with dgx.Solver(c.mesh, c.params) as s:
            s.tile = tile
            s.set_state(c.U0)
            _, f = s.residual()
            n = s.step(c.dt, c.scheme, 3)
            got[tile] = (f, n, s.get_state())
    e = (rel(got[1][0], got[0][0]), float(np.max(np.abs(got[1][1] / got[0][1] - 1.0))),
         rel(got[1][2], got[0][2]))
    print(name, "f %.2e norms %.2e state %.2e" % e, flush=True)
    assert e[0] < 1e-12 and e[1] < 1e-12 and e[2] < 1e-13


@pytest.mark.parametrize("name", ["p1_stretched_walls_3x3x3", "p3_channel_3x1x3"])
def test_switching_kernels_between_steps(name):
    """A step of the tiled kernel leaves no trace records: the one-row kernel
    and the residual adjoint that follow recompute them."""
    c = CASES[name]()
    w = np.random.default_rng(9).standard_normal(c.U0.size)
    got = []
    for tiles in ((0, 0, 0), (1, 0, 1)):
        with dgx.Solver(c.mesh, c.params) as s:
            s.set_state(c.U0)
            for t in tiles:
                s.tile = t
                s.step(c.dt, c.scheme, 1, norms=False)
            got.append((s.get_state(), s.residual_vjp(w)))
    assert rel(got[1][0], got[0][0]) < 1e-13
    assert rel(got[1][1], got[0][1]) < 1e-11  # (df/dU)^T w amplifies the state's difference
