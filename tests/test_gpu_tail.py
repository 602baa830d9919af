"""The small levels of a V-cycle in one block against the separate kernels, on
whole FGMRES solves: the same bits and iteration counts."""
import numpy as np
import pytest

from helpers import cases, channel_pair, vfs

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


def _box(cells):
    """A box without periodic directions: slip sides, inlet and outlet."""
    c = cases.box_flow(*cells)
    ctx = vfs.Context(cases.params_for(vfs, c, 1e-2, les=0))
    ctx.upload("COOR", c.coor)
    ctx.form_metrics()
    ctx.upload("UCONT", c.ucont)
    return ctx


@pytest.mark.parametrize("form", ["compact", "full", "fp64"])
@pytest.mark.parametrize("grid", ["blanked", "box", "blanked-box"])
@pytest.mark.parametrize("cells", [(16, 12, 16), (17, 7, 19), (24, 16, 20), (68, 32, 68)], ids=str)
def test_one_block_row_masks_bitwise(monkeypatch, cells, grid, form):
    """The same with points that are no rows: blanked cells (whose coarse cells
    are rows as long as one child is) and ghosts that nothing wraps to.  A
    fixed number of iterations: blanked grids converge slowly."""
    monkeypatch.setenv("VFS_SMOOTH_COMPACT", "0" if form == "full" else "1")
    out = []
    for tail in ("1", "0"):
        monkeypatch.setenv("VFS_MG_TAIL", tail)
        ctx = _box(cells) if "box" in grid else channel_pair(*cells, les=0)[2]
        with ctx:
            ctx.poisson_rhs()
            if "blanked" in grid:
                nv = np.zeros(ctx.field_shape("NVERT"))
                nv[2:5, 3:6, 4:9] = 1.0
                ctx.upload("NVERT", nv)
            ctx.upload("PHI", np.zeros(ctx.field_shape("PHI")))
            opts = vfs.default_solve_opts(tol=1e-9, use_guess=0, maxit=12, mg_fp32=0 if form == "fp64" else 1)
            st = ctx.poisson_solve(opts, check=False)
            out.append((st.iterations, ctx.download("PHI")))
    assert np.isfinite(out[0][1]).all() and np.abs(out[0][1]).max() > 0
    assert out[0][0] == out[1][0]
    assert np.array_equal(out[0][1], out[1][1])
