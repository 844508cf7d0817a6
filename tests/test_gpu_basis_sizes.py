"""State conversions at the sizes and orders where the kernel changes: several
elements per workgroup at p <= 2 (full, partly filled and single workgroups), a
line of nodes per lane on large meshes, and the mixed forms' sums.

Bar: as test_gpu_basis; the mixed forms round once more per term of the three
sums of p + 1 terms."""
import time

import numpy as np
import pytest

from dgpr_amd import dgx
from test_gpu_basis import norm_bound

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

SIZES = {
    0: [(1, 1, 1), (64, 1, 1), (13, 5, 1)],
    1: [(7, 1, 1), (8, 1, 1), (3, 3, 1), (131, 17, 11), (131, 17, 12)],  # lines from 24576
    2: [(1, 1, 1), (2, 1, 1), (3, 1, 1), (29, 16, 23), (29, 16, 24)],    # from 10923
    3: [(2, 1, 1), (17, 27, 26), (17, 27, 27)],                          # from 12288
}


def solver(p, n, precision):
    mesh = dgx.Mesh(p, 1, *n, [dgx.PERIODIC] * 6, dgx.box_nodes(1, *n, 0, 0, 0, 1, 1, 1, 0.0, 1))
    s = dgx.Solver(mesh, dgx.make_reference_state(mu=1e-3, c=1.0, u=0.2))
    s.precision = precision
    return s


@pytest.mark.parametrize("precision", ["fp64", "mixed_records"])
@pytest.mark.parametrize("p", sorted(SIZES))
def test_round_trip(p, precision):
    bar = 2.0 ** -53 * norm_bound(p) * (1 if precision == "fp64" else 1 + 3 * (p + 1))
    for n in SIZES[p]:
        with solver(p, n, precision) as s:
            rng = np.random.default_rng(p)
            U = rng.standard_normal((s.nelem, 5, s.nbf)) * 10.0 ** rng.integers(-6, 7, (s.nelem, 5, 1))
            s.set_state(U.reshape(-1))
            got = s.get_state().reshape(U.shape)
        err = (np.abs(got - U).max(axis=2) / np.abs(U).max(axis=2)).max()
        print("p", p, precision, n, "%.2e of %.2e" % (err, bar), flush=True)
        assert err <= bar


def test_mixed_conversion_fills_its_lanes():
    """64^3 p = 1: at most twice as long as in FP64 (5.4 times with one 8-node element
    per 64-lane workgroup)."""
    us = {}
    for precision in ("fp64", "mixed"):
        with solver(1, (64, 64, 64), precision) as s:
            U = torch.ones(s.nstate, dtype=torch.float64, device="cuda")
            torch.cuda.synchronize()
            best = 1e9
            for _ in range(6):
                t = time.perf_counter()
                for _ in range(40):
                    s.set_state_device(U.data_ptr())
                best = min(best, (time.perf_counter() - t) / 40 * 1e6)
            us[precision] = best
    print("set_state_device us:", us, flush=True)
    assert us["mixed"] < 2.0 * us["fp64"]
