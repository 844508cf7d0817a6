"""The tiled stage kernel with a line of nodes per lane (FP64, p = 2 and 3)
against the one-row kernel: tiles of 7 (p = 2) and 4 (p = 3) elements, full,
partly filled and of one element; at p = 3 the kernel takes over at 12288
elements, and runs every tiled ensemble unit.  Its step, trace records (read
by the adjoint) and fused norms, and the mesh sizes from which p = 2 uses it.

Bars (the same sums in another order): f to a hundred roundings of its largest
terms, of size max|U| (|u| + c) (2p+1) / h (f itself can be 1e-5 of them: the
one-row and the general-order kernel differ by 1e-11 of f on the 24x16x32
channel); norms 1e-12; state after three steps 1e-13; gradients amplify the
state's difference, 1e-11.
"""
import numpy as np
import pytest

from dgpr_amd import dgx
from test_gpu_parity import DEFAULT_BOUNDS, rel
from test_gpu_tile import channel, stretched_case

pytestmark = pytest.mark.gpu

PER = [dgx.PERIODIC] * 6
CASES = {
    "p2_stretched_1x1x1": lambda: stretched_case(2, (1, 1, 1), PER, 1),
    "p2_stretched_7x1x1": lambda: stretched_case(2, (7, 1, 1), PER, 2),
    "p2_stretched_walls_3x3x3": lambda: stretched_case(2, (3, 3, 3), DEFAULT_BOUNDS, 3),
    "p2_channel_4x2x1": lambda: channel(2, (4, 2, 1), 4),
    "p2_channel_3x5x4": lambda: channel(2, (3, 5, 4), 5),
    "p3_stretched_walls_17x27x27": lambda: stretched_case(3, (17, 27, 27), DEFAULT_BOUNDS, 6),
    "p3_channel_24x16x32": lambda: channel(3, (24, 16, 32), 7),
}


def rates(c):
    """(|u| + c) (2p+1) / h, the largest terms of f over max|U|, and that plus the
    viscous rate eta mu ((2p+1) / h)^2: about 1 / dt at the stability limit."""
    X = c.mesh.nodes.reshape(-1, 8, 3)
    k = (2 * c.mesh.p + 1) / min(np.abs(X[:, 1 << d, d] - X[:, 0, d]).min() for d in range(3))
    wave = (np.abs(c.params.Ufr[1] / c.params.Ufr[0]) + c.params.c) * k
    return wave, wave + c.params.eta * c.params.mu * k * k


@pytest.mark.parametrize("name", sorted(CASES))
def test_line_tile_against_one_row(name):
    c = CASES[name]()
    w = np.random.default_rng(9).standard_normal(c.U0.size)
    wave, rate = rates(c)
    dt = min(c.dt, 0.02 / rate)
    got = {}
    for tile in (0, 1):
        with dgx.Solver(c.mesh, c.params) as s:
            s.tile = tile
            s.set_state(c.U0)
            _, f = s.residual()
            n = s.step(dt, c.scheme, 3)
            got[tile] = (f, n, s.get_state(), s.residual_vjp(w))
    df = np.abs(got[1][0] - got[0][0]).max() / (np.abs(c.U0).max() * wave)
    e = (df, float(np.max(np.abs(got[1][1] / got[0][1] - 1.0))),
         rel(got[1][2], got[0][2]), rel(got[1][3], got[0][3]))
    print(name, "f %.2e norms %.2e state %.2e vjp %.2e" % e, flush=True)
    assert e[0] < 100 * 2.0 ** -53 and e[1] < 1e-12 and e[2] < 1e-13 and e[3] < 1e-11


def test_line_tile_adjoint_records():
    """The adjoint's forward sweep on the tiled kernel writes every face's record."""
    c = stretched_case(2, (3, 3, 3), DEFAULT_BOUNDS, 8)
    got = []
    for tile in (0, 1):
        with dgx.Solver(c.mesh, c.params) as s:
            s.tile = tile
            s.set_state(c.U0)
            got.append(s.adjoint_rk4(c.dt, 3))
    assert rel(got[1][1], got[0][1]) < 1e-11 and abs(got[1][2] / got[0][2] - 1.0) < 1e-9


@pytest.mark.parametrize("affine", [True, False])
def test_line_tile_ensemble(affine):
    """The units of every order that tuning picks: tiled ones with the large members,
    and then members of less than a tile to several tiles."""
    sizes = [(1, 1, 1), (3, 1, 1), (2, 2, 2), (3, 3, 1), (19, 17, 16)]
    cs = [stretched_case(p, n, PER, 10 * p + i) if affine else channel(p, n, 10 * p + i)
          for p in (1, 2, 3) for i, n in enumerate(sizes)]
    dts = [min(c.dt, 0.02 / rates(c)[1]) for c in cs]
    ref = []
    for c, dt in zip(cs, dts):
        with dgx.Solver(c.mesh, c.params) as s:
            s.tile = 0
            s.set_state(c.U0)
            s.step(dt, "RK4", 2, norms=False)
            ref.append(s.get_state())
    with dgx.Ensemble([c.mesh for c in cs], [c.params for c in cs]) as en:
        for m, c in zip(en.members, cs):
            m.set_state(c.U0)
        en.autotune("RK4", dts)
        for m, c in zip(en.members, cs):
            m.set_state(c.U0)
        en.step("RK4", dts, 2)
        err = max(rel(m.get_state(), r) for m, r in zip(en.members, ref))
        print("ensemble %.2e tiles" % err, [en.member_tuning(i)[1] for i in range(len(cs))],
              flush=True)
    assert err < 1e-13


@pytest.mark.parametrize("curved, n, tile", [(False, (32, 32, 15), 0), (False, (32, 32, 16), 1),
                                             (True, (16, 16, 31), 0), (True, (16, 16, 32), 1)])
def test_p2_default_tile(curved, n, tile):
    c = channel(2, n, 1) if curved else stretched_case(2, n, PER, 1)
    with dgx.Solver(c.mesh, c.params) as s:
        assert s.tile == tile and s.stage_waves == 2
