"""Device memory that contexts keep and can do without (dgx_pool.cpp), on the
CPU against a stand-in for the HIP runtime (tests/cpu/pool_check.cpp, and
tests/cpu/memory_limit_check.cpp with contexts at the limit of the memory), and
overlapping adjoint calls on one solver on the GPU."""
import os
import subprocess
import threading

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("program, sources", [
    ("pool_check", ["dgx_pool"]),
    ("memory_limit_check", ["dgx_pool", "dgx_api", "dgx_tables", "dgx_host"]),
])
def test_on_the_cpu(program, sources, tmp_path):
    exe = str(tmp_path / program)
    csrc = os.path.join(ROOT, "dgpr_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread",
                    "-I" + os.path.join(ROOT, "tests", "cpu", "pool"), "-I" + csrc,
                    "-I" + os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "cpu", program + ".cpp")]
                   + [os.path.join(csrc, s + ".cpp") for s in sources] + ["-o", exe],
                   check=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.gpu
def test_overlapping_products_of_one_solver():
    """Vector-Jacobian products of four threads on one solver: each its own."""
    from dgpr_amd import cases, dgx
    c = cases.channel_case(6, 5, 4, p=2, seed=3, nsteps=1)
    w = [np.random.default_rng(t).standard_normal(c.U0.size) for t in range(4)]
    with dgx.Solver(c.mesh, c.params) as s:
        s.set_state(c.U0)
        ref = [s.residual_vjp(x) for x in w]
        bad = []

        def work(t):
            for _ in range(20):
                if not np.array_equal(s.residual_vjp(w[t]), ref[t]):
                    bad.append(t)

        threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not bad
