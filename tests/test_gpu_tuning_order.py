"""Occupancy targets, tiles and precisions chosen in any order leave a stage
kernel that exists: a step after each call, equal to the one-row kernel's."""
import itertools

import numpy as np
import pytest

from dgpr_amd import cases, dgx
from test_gpu_parity import rel

pytestmark = pytest.mark.gpu


def reference(c):
    with dgx.Solver(c.mesh, c.params) as s:
        s.tile = 0
        s.set_state(c.U0)
        s.step(c.dt, c.scheme, 1, norms=False)
        return s.get_state()


@pytest.mark.parametrize("p, n", [(1, (4, 3, 3)), (2, (4, 3, 3)), (2, (32, 32, 16)), (3, (4, 3, 3))])
def test_every_order_of_calls_steps(p, n):
    c = cases.tgv_case(nxyz=n, p=p, seed=p, M=0.3)
    ref = reference(c)
    acts = {
        "mixed": lambda s: setattr(s, "precision", "mixed"),
        "fp64": lambda s: setattr(s, "precision", "fp64"),
        "waves1": lambda s: setattr(s, "stage_waves", 1),
        "waves3": lambda s: setattr(s, "stage_waves", 3),
        "tile0": lambda s: setattr(s, "tile", 0),
        "tile1": lambda s: setattr(s, "tile", 1),
        "autotune": lambda s: s.autotune(1),
    }
    for seq in itertools.permutations(acts, 3 if c.mesh.nelem < 100 else 2):
        with dgx.Solver(c.mesh, c.params) as s:
            for a in seq:
                try:
                    acts[a](s)
                except dgx.DgxError:
                    # a target of 1 with the tiled kernel: the order's default or chosen
                    assert a == "waves1" and s.tile == 1
                    assert p == 3 or "tile1" in seq
                s.set_state(c.U0)
                s.step(c.dt, c.scheme, 1, norms=False)
                got = s.get_state()
            # FP32 records: their rounding times dt f, 1e-6 of the state at most
            assert rel(got, ref) < (1e-13 if s.precision == "fp64" else 1e-6), seq


@pytest.mark.parametrize("p, n", [(1, (3, 3, 3)), (2, (32, 32, 16))])
def test_target_of_one_on_a_new_context(p, n):
    """Accepted where the tile is a default; the default comes back with the target."""
    c = cases.tgv_case(nxyz=n, p=p, seed=p, M=0.3)
    with dgx.Solver(c.mesh, c.params) as s:
        assert s.tile == 1
        s.stage_waves = 1
        assert (s.tile, s.stage_waves) == (0, 1)
        s.set_state(c.U0)
        n1 = s.step(c.dt, c.scheme, 2)
        s.stage_waves = 2
        assert (s.tile, s.stage_waves) == (1, 2)
        n2 = s.step(c.dt, c.scheme, 1)
        assert np.isfinite(n1).all() and np.isfinite(n2).all()


def test_precision_round_trip_with_a_target_of_one():
    c = cases.tgv_case(nxyz=(3, 3, 3), p=1, seed=2, M=0.3)
    ref = reference(c)
    with dgx.Solver(c.mesh, c.params) as s:
        s.precision = "mixed"
        s.stage_waves = 1
        s.precision = "fp64"
        s.set_state(c.U0)
        s.step(c.dt, c.scheme, 1, norms=False)
        assert rel(s.get_state(), ref) < 1e-13


@pytest.mark.parametrize("p, n", [(1, 32), (2, 32), (3, 16), (3, 32)])
def test_a_target_of_three_is_no_trap(p, n):
    """No target of the FP64 tiled kernel needs half as long again as another (with
    spilled registers a target of 3 needed 2.4 times as long)."""
    c = cases.tgv_case(n=n, p=p, M=0.3)
    with dgx.Solver(c.mesh, c.params) as s:
        s.tile = 1
        s.set_state(c.U0)
        s.autotune(20)
        _, us = s.autotune(50)
        print("p %d n %d us at 2 and 3 waves:" % (p, n), us[1:], flush=True)
        assert us[2] < 1.5 * us[1]
