"""Meshes on which the two elements at a face do not have the same face: the two
sides of a periodic direction curved differently.  Every kernel takes the
neighbour's gradient with the neighbour's own geometry, so the tiled kernels
agree with the one-row and the general-order kernel there too.

Bars as test_gpu_tile (the same sums in another order): f 1e-12 and the state
after three steps 1e-13 relative, norms and gradients 1e-12 and 1e-11.
"""
import numpy as np
import pytest

from dgpr_amd import cases, dgx
from test_gpu_parity import DEFAULT_BOUNDS, perturbed_uniform, rel
from test_gpu_tile import channel, stretched_case

pytestmark = pytest.mark.gpu


def unmatched_case(p, nxyz, bounds, seed):
    """Curved box: the nodes of the side x = 0 (and, where z is periodic, z = 0) are
    displaced along the side, those of the opposite side are not."""
    c = stretched_case(p, nxyz, bounds, seed)
    nx, ny, nz = nxyz
    X = c.mesh.nodes.reshape(nz, ny, nx, 2, 2, 2, 3).copy()
    h = 2.0 / max(nxyz)
    y, z = X[:, :, 0, :, :, 0, 1].copy(), X[:, :, 0, :, :, 0, 2].copy()
    inside = np.sin(0.5 * np.pi * y)  # walls stay where they are
    X[:, :, 0, :, :, 0, 1] += 0.15 * h * inside * np.cos(0.5 * np.pi * z)
    X[:, :, 0, :, :, 0, 0] += 0.1 * h * inside
    if bounds[4] == dgx.PERIODIC:
        x = X[0, :, :, 0, :, :, 0].copy()
        X[0, :, :, 0, :, :, 2] += 0.1 * h * np.sin(np.pi * x)
    mesh = dgx.Mesh(p, 1, nx, ny, nz, bounds, X)
    assert not mesh.affine
    return cases.Case("unmatched", mesh, c.params, perturbed_uniform(mesh, c.params, 0.03, seed),
                      "RK4", 2e-3, 3)


WALLS_Y = [dgx.PERIODIC, dgx.PERIODIC, dgx.NO_SLIP_WALL, dgx.NO_SLIP_WALL, dgx.PERIODIC,
           dgx.PERIODIC]
CASES = {
    "p1_3x3x3": lambda: unmatched_case(1, (3, 3, 3), WALLS_Y, 1),
    "p2_5x3x1": lambda: unmatched_case(2, (5, 3, 1), WALLS_Y, 2),
    "p3_3x3x3": lambda: unmatched_case(3, (3, 3, 3), WALLS_Y, 3),
    "p3_1x3x2": lambda: unmatched_case(3, (1, 3, 2), [dgx.PERIODIC] * 6, 4),
}


def run(c, tile, waves=None):
    with dgx.Solver(c.mesh, c.params) as s:
        s.tile = tile
        if waves:
            s.stage_waves = waves
        assert not s.faces_match
        s.set_state(c.U0)
        _, f = s.residual()
        n = s.step(c.dt, c.scheme, 3)
        g = s.residual_vjp(np.cos(np.arange(c.U0.size)))
        J = s.adjoint_rk4(c.dt, 2)
        return f, n, s.get_state(), g, J[1]


@pytest.mark.parametrize("waves", [2, 3])
@pytest.mark.parametrize("name", sorted(CASES))
def test_tiled_kernel(name, waves):
    c = CASES[name]()
    ref, got = run(c, 0), run(c, 1, waves)
    e = (rel(got[0], ref[0]), float(np.max(np.abs(got[1] / ref[1] - 1.0))), rel(got[2], ref[2]),
         rel(got[3], ref[3]), rel(got[4], ref[4]))
    print(name, "f %.2e norms %.2e state %.2e vjp %.2e adjoint %.2e" % e, flush=True)
    assert e[0] < 1e-12 and e[1] < 1e-12 and e[2] < 1e-13 and e[3] < 1e-11 and e[4] < 1e-11


def test_line_tile_sizes():
    """At a size from which matched meshes run the kernel with a line of nodes per lane."""
    for p, n in ((3, (24, 23, 23)), (2, (24, 21, 17))):
        c = unmatched_case(p, n, WALLS_Y, 5)
        f = []
        for tile in (0, 1):
            with dgx.Solver(c.mesh, c.params) as s:
                assert s.tile == (1 if p == 3 else 0)  # p = 2: matched ones tile from 8192
                s.tile = tile
                s.set_state(c.U0)
                f.append(s.residual()[1])
        assert rel(f[1], f[0]) < 1e-11  # |f| is small against its terms on fine meshes


def test_ensemble():
    """Tuned units of mixed members; unmatched ones keep to record-reading units."""
    cs = [CASES[n]() for n in sorted(CASES)] + [channel(p, (19, 17, 16), p) for p in (1, 2, 3)]
    ref = []
    for c in cs:
        with dgx.Solver(c.mesh, c.params) as s:
            s.tile = 0
            s.set_state(c.U0)
            s.step(c.dt, "RK4", 2, norms=False)
            ref.append(s.get_state())
    with dgx.Ensemble([c.mesh for c in cs], [c.params for c in cs]) as en:
        dts = [c.dt for c in cs]
        en.autotune("RK4", dts)
        for m, c in zip(en.members, cs):
            m.set_state(c.U0)
        en.step("RK4", dts, 2)
        assert max(rel(m.get_state(), r) for m, r in zip(en.members, ref)) < 1e-13


def test_generated_meshes_match():
    """The meshes of the generators, curved and with coordinates far from the origin."""
    for c in (cases.tgv_case(n=4, p=1, amp=0.1), channel(2, (5, 3, 4), 1),
              stretched_case(3, (3, 2, 2), DEFAULT_BOUNDS, 2)):
        for shift in (0.0, 1e3 / 3.0):
            mesh = dgx.Mesh(c.mesh.p, 1, c.mesh.nx, c.mesh.ny, c.mesh.nz, c.mesh.bounds,
                            c.mesh.nodes + shift)
            with dgx.Solver(mesh, c.params) as s:
                assert s.faces_match
