"""State conversions between the reference basis and the Gauss nodes: the round
trip of set_state and get_state at every order, on small meshes and, at p = 1 to 3,
on one large enough for the kernel with a line of nodes per lane, with a partly
filled last block.

Bar: both conversions are formed in double-double and rounded once, so with
B the 1D matrix and u = 2^-53 the nodal values err by u |V|, |V| <= |B|^3 |U| (row
sum norms), and the state by u (|B^-1|^3 |B|^3 + 1) max|U|.
"""
import numpy as np
import pytest

from dgpr_amd import dgx

pytestmark = pytest.mark.gpu


def norm_bound(p):
    """(|B|_inf |B^-1|_inf)^3 + 1, B[i][j] the equispaced Lagrange basis at Gauss node i."""
    g = 0.5 * (np.polynomial.legendre.leggauss(p + 1)[0] + 1.0)
    x = np.linspace(0.0, 1.0, p + 1) if p else np.array([0.5])
    B = np.array([[np.prod([(t - x[m]) / (x[j] - x[m]) for m in range(p + 1) if m != j])
                   for j in range(p + 1)] for t in g])
    return (np.abs(B).sum(1).max() * np.abs(np.linalg.inv(B)).sum(1).max()) ** 3 + 1.0


@pytest.mark.parametrize("p", range(9))
def test_state_round_trip(p):
    large = {1: [(131, 17, 8)], 2: [(29, 16, 16)], 3: [(17, 17, 15)]}
    for n in [(1, 1, 1), (5, 3, 1), (17, 1, 1)] + large.get(p, []):
        mesh = dgx.Mesh(p, 1, *n, [dgx.PERIODIC] * 6, dgx.box_nodes(1, *n, 0, 0, 0, 1, 1, 1, 0.0, 1))
        prm = dgx.make_reference_state(mu=1e-3, c=1.0, u=0.2)
        rng = np.random.default_rng(p)
        U = rng.standard_normal((mesh.nelem, 5, mesh.nbf)) * 10.0 ** rng.integers(-6, 7, (mesh.nelem, 5, 1))
        with dgx.Solver(mesh, prm) as s:
            s.set_state(U.reshape(-1))
            got = s.get_state().reshape(U.shape)
        err = np.abs(got - U).max(axis=2) / np.abs(U).max(axis=2)
        print("p", p, n, "%.2e of %.2e" % (err.max(), 2.0 ** -53 * norm_bound(p)), flush=True)
        assert err.max() <= 2.0 ** -53 * norm_bound(p)
