"""Curved geometry evaluated in the kernels against the stored one, in every
form that a mesh without the room for the store takes.

Bars: the two give the same values to a few roundings of the geometry, so f
agrees to 1e-12 of its size, norms to 1e-12, the state after three steps to
1e-13, gradients to 1e-11; in the mixed forms a last bit can flip the rounding of
an FP32 record (2^-24 of a trace), 1e-5 of f.
"""
import numpy as np
import pytest

from dgpr_amd import cases, dgx
from test_gpu_parity import rel

pytestmark = pytest.mark.gpu

ORDERS = [(1, 2), (2, 2), (3, 2), (1, 3), (3, 3), (0, 1), (0, 2), (2, 5), (4, 1), (4, 2), (5, 3),
          (8, 1), (8, 8)]


def channel(p, q, seed=1):
    return cases.channel_case(3, 2, 2, p=p, q=q, seed=seed, nsteps=3)


def run(c, stored, precision):
    with dgx.Solver(c.mesh, c.params) as s:
        assert s.stored_geometry
        s.stored_geometry = stored
        s.precision = precision
        s.set_state(c.U0)
        R, f = s.residual()
        n = s.step(c.dt, c.scheme, 3)
        assert s.stored_geometry == stored
        out = [f, R, n, s.get_state()]
        if precision == "fp64" and 1 <= c.mesh.p <= 3 and c.mesh.q <= 3:
            out.append(s.residual_vjp(np.cos(np.arange(c.U0.size))))
        return out


@pytest.mark.parametrize("precision", ["fp64", "mixed_records"])
@pytest.mark.parametrize("p, q", ORDERS)
def test_evaluated_against_stored(p, q, precision):
    c = channel(p, q)
    bars = [1e-12, 1e-12, 1e-12, 1e-13, 1e-11] if precision == "fp64" else [1e-5, 1e-5, 1e-5, 1e-6]
    ref, got = run(c, True, precision), run(c, False, precision)
    e = [rel(g, r) for g, r in zip(got, ref)]
    print("p %d q %d %s" % (p, q, precision), ["%.1e" % x for x in e], flush=True)
    assert all(x < b for x, b in zip(e, bars))


def test_switching_between_steps():
    c = channel(2, 2)
    got = []
    for flags in ((True,) * 4, (False, True, False, True)):
        with dgx.Solver(c.mesh, c.params) as s:
            s.set_state(c.U0)
            for f in flags:
                s.stored_geometry = f
                s.step(c.dt, c.scheme, 1, norms=False)
            got.append(s.get_state())
    assert rel(got[1], got[0]) < 1e-13


def test_meshes_that_store_none():
    for c in (cases.tgv_case(n=2, p=2), cases.tgv_case(n=2, p=5), cases.channel_case(3, 2, 2, p=3)):
        with dgx.Solver(c.mesh, c.params) as s:
            assert not s.stored_geometry
            s.stored_geometry = False
            with pytest.raises(dgx.DgxError) as ei:
                s.stored_geometry = True
            assert ei.value.status == dgx.ERR_UNSUPPORTED


def test_ensemble_keeps_what_it_reads():
    """General-order members read the store from the ensemble's tables, the batched
    orders do not."""
    cs = [channel(2, 2), channel(4, 2), channel(4, 1, 2)]
    ref = []
    for c in cs:
        with dgx.Solver(c.mesh, c.params) as s:
            s.set_state(c.U0)
            s.step(c.dt, "RK4", 2, norms=False)
            ref.append(s.get_state())
    with dgx.Ensemble([c.mesh for c in cs], [c.params for c in cs]) as en:
        dts = [c.dt for c in cs]
        for m, c in zip(en.members, cs):
            m.set_state(c.U0)
        en.step("RK4", dts, 1)
        en.members[0].stored_geometry = False
        with pytest.raises(dgx.DgxError, match="in use"):
            en.members[1].stored_geometry = False
        en.step("RK4", dts, 1)
        for m, r in zip(en.members, ref):
            assert rel(m.get_state(), r) < 1e-13
