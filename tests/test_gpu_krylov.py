"""The Gram-Schmidt sweeps with their sums finished by the last block: every
basis-size instance (4, 8, 16, 32 vectors) on grids from a handful of blocks to
more than the partials hold, checked with the oracle's operator."""
import os
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

from helpers import channel_pair, vfs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("restart", [3, 7, 15, 31])
@pytest.mark.parametrize("cells", [(4, 4, 6), (17, 11, 13), (96, 64, 80)], ids=str)
def test_restart_lengths(cells, restart):
    """A weak preconditioner (one level, one sweep) fills the basis; the
    residual the solver reports is the one of its solution (the recurrences'
    rounding is far below the tolerance)."""
    c, o, ctx = channel_pair(*cells, les=0)
    with ctx:
        o.poisson_rhs()
        ctx.poisson_rhs()
        ctx.upload("PHI", np.zeros(o.shape))
        opts = vfs.default_solve_opts(tol=1e-6, use_guess=0, levels=1, coarse_sweeps=1, restart=restart, maxit=40)
        st = ctx.poisson_solve(opts, check=False)
        r = np.linalg.norm(o["b"] - o.poisson_apply(ctx.download("PHI"))) / np.linalg.norm(o["b"])
        assert abs(r - st.relres) <= 1e-9
        assert r < 0.9 and (st.relres <= 1e-6 or st.iterations == 40)
        st2 = ctx.poisson_solve(opts, check=False)  # the counters are back at zero: the same bits again
        assert (st2.iterations, st2.relres) == (st.iterations, st.relres)


@pytest.mark.parametrize("tol", [1e-12, 1e-18])
@pytest.mark.parametrize("cells", [(4, 4, 6), (8, 6, 8)], ids=str)
def test_exhausted_basis(cells, tol):
    """A preconditioner that is the inverse (an algebraic hierarchy of one
    level) leaves nothing but rounding of the first new vector.  Its norm is then
    the small difference the second pass computes it as, and may come out as
    zero: the solve stops at the residual a double can reach, finite, also when
    it is asked for less.  96 and 384 rows, condition numbers 45 and 85: rows x
    2^-53 x condition number is 4e-12 at most."""
    c, o, ctx = channel_pair(*cells, les=0)
    with ctx:
        o.poisson_rhs()
        ctx.poisson_rhs()
        ctx.upload("PHI", np.zeros(o.shape))
        st = ctx.poisson_solve(vfs.default_solve_opts(tol=tol, use_guess=0, amg=1, maxit=12), check=False)
        phi = ctx.download("PHI")
        assert np.isfinite(phi).all()
        r = np.linalg.norm(o["b"] - o.poisson_apply(phi)) / np.linalg.norm(o["b"])
        assert r <= 1e-11
        assert st.iterations <= (2 if tol == 1e-12 else 12)


SCALARS = """
from helpers import channel_pair, vfs
c, o, ctx = channel_pair(17, 11, 13, les=0)
ctx.poisson_rhs()
st = ctx.poisson_solve(vfs.default_solve_opts(tol=1e-8, use_guess=0))
out = [ctx.min_dt(), ctx.calc_k_flux(), ctx.divergence(), st.iterations, st.relres]
ctx.close()
"""


def test_host_results_without_coherent_default():
    """The scalars the host polls for arrive where the runtime's default host
    memory is not coherent (a process of its own: the setting is read at its
    start), with the bits they have otherwise."""
    here = {}
    exec(SCALARS, here)
    tests = Path(__file__).resolve().parent
    env = dict(os.environ, HIP_HOST_COHERENT="0",
               PYTHONPATH=os.pathsep.join(str(p) for p in (tests, tests.parent, tests.parent / "oracle")))
    r = subprocess.run([sys.executable, "-c", SCALARS + "print('SCALARS', *map(float.hex, map(float, out)))"], env=env,
                       cwd=tests.parent, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    got = r.stdout.split("SCALARS")[1].split()
    assert got == [float(v).hex() for v in here["out"]]
