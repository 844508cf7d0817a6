"""States without a real sound speed or density: the residual has no finite
value there, whichever form of the Roe flux a kernel takes, so that a run that
has left the admissible states is reported (DGX_ERR_NAN) and not continued."""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_roe_flux_forms(tmp_path):
    """roe_flux_fp64 against roe_flux on the CPU (tests/cpu/roe_check.cpp)."""
    exe = str(tmp_path / "roe_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wno-unknown-pragmas",
                    "-I" + os.path.join(ROOT, "tests", "cpu"),
                    "-I" + os.path.join(ROOT, "dgpr_amd", "csrc"),
                    "-I" + os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "cpu", "roe_check.cpp"), "-o", exe],
                   check=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("p, tile", [(1, 0), (1, 1), (2, 0), (2, 1), (3, 0), (3, 1), (3, 2), (4, 2)])
def test_negated_state_is_refused(p, tile):
    """Every density and energy negative: each face has two negative densities."""
    from dgpr_amd import cases, dgx
    c = cases.tgv_case(n=3, p=p, M=0.3)
    with dgx.Solver(c.mesh, c.params) as s:
        s.tile = tile
        s.set_state(-c.U0)
        _, f = s.residual()
        assert not np.isfinite(f).all()
        with pytest.raises(dgx.DgxError, match="unstable"):
            s.step(1e-4, "RK4", 1)
