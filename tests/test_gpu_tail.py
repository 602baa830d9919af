"""The small levels of a V-cycle in one block against the separate kernels, on
whole FGMRES solves: the same bits and iteration counts."""
import numpy as np
import pytest

from helpers import channel_pair, vfs

pytestmark = pytest.mark.gpu

# whole hierarchies in one block (coarsenable, single odd level, one line
# segment), the coarse levels only, and no level small enough but the last
CELLS = [(16, 12, 16), (17, 11, 13), (4, 4, 6), (24, 16, 20), (40, 24, 36), (64, 48, 64), (36, 70, 44)]
# odd periodic counts with one segment per line: lines of one colour, held by
# different wavefronts, read each other's values from before the half-sweep (the
# last grid on its coarsest level, 17x8x17, which has too many rows for a dense solve)
CELLS += [(17, 7, 19), (16, 8, 17), (17, 8, 17), (19, 6, 16), (68, 32, 68)]


@pytest.mark.parametrize("form", ["compact", "full", "fp64", "deep"])
@pytest.mark.parametrize("cells", CELLS, ids=str)
def test_one_block_levels_bitwise(monkeypatch, form, cells):
    monkeypatch.setenv("VFS_SMOOTH_COMPACT", "0" if form == "full" else "1")
    kw = {"mg_fp32": 0} if form == "fp64" else {"deep_level": 1, "deep_pre": 0, "deep_post": 1} if form == "deep" else {}
    out = []
    for tail in ("1", "0"):
        monkeypatch.setenv("VFS_MG_TAIL", tail)
        c, o, ctx = channel_pair(*cells, les=0)
        with ctx:
            ctx.poisson_rhs()
            opts = vfs.default_solve_opts(tol=1e-9, use_guess=0, maxit=400, **kw)
            for _ in range(2):  # the second solve replays what the first captured
                ctx.upload("PHI", np.zeros(o.shape))
                st = ctx.poisson_solve(opts)
            out.append((st.iterations, ctx.download("PHI")))
    assert out[0][0] == out[1][0]
    assert np.array_equal(out[0][1], out[1][1])
