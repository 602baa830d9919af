"""The k-marching passes choose the planes per block by the grid: runs of one
plane on small grids, runs that do not divide the plane count and long runs,
against the oracle."""
import numpy as np
import pytest

from helpers import channel_pair, relerr

pytestmark = pytest.mark.gpu

# relative to the field's maximum: a value is a sum of tens of terms of its
# neighbourhood's size, each rounded to 2^-53
TOL = 1e-12


@pytest.mark.parametrize("second_order", [1, 0])
@pytest.mark.parametrize("cells", [(4, 4, 4), (33, 17, 19), (66, 34, 131), (160, 96, 70)], ids=str)
def test_run_lengths(cells, second_order):
    c, o, ctx = channel_pair(*cells, les=1, second_order=second_order)
    with ctx:
        o.eddy_viscosity()
        ctx.eddy_viscosity()
        assert relerr(ctx.download("NU_T"), o["nu_t"]) <= TOL
        o.formfunction2(1.0)
        ctx.formfunction2(1.0)
        assert relerr(ctx.download("RHS"), o["rhs"]) <= TOL
        o.runge_kutta()
        ctx.runge_kutta()
        assert relerr(ctx.download("UCONT"), o["ucont"]) <= TOL


@pytest.mark.parametrize("blank", [0, 1], ids=["open", "blanked"])
@pytest.mark.parametrize("laplacian,les", [(1, 1), (0, 1), (1, 0)])
@pytest.mark.parametrize("cells", [(31, 7, 5), (32, 8, 6), (33, 9, 7), (65, 15, 4)], ids=str)
def test_face_tile_edges(monkeypatch, cells, laplacian, les, blank):
    """The fused face pass at the edges of its 32 x 8 tiles, against the oracle
    and, to the bit, against the pass that stores the flux planes."""
    c, o, ctx = channel_pair(*cells, les=les, laplacian=laplacian)
    with ctx:
        if blank:
            nv = np.zeros(o.shape)
            nv[2:4, 3:5, 4:7] = 1.0
            o.m["nvert"][...] = nv
            ctx.upload("NVERT", nv)
        if les:
            o.eddy_viscosity()
            ctx.upload("NU_T", o["nu_t"])
        o.formfunction2(1.0)
        out = []
        for fused in ("1", "0"):
            monkeypatch.setenv("VFS_FUSED_FP", fused)
            ctx.upload("RHS", np.zeros(o["rhs"].shape))
            ctx.formfunction2(1.0)
            out.append(ctx.download("RHS"))
        assert np.abs(out[0]).max() > 0
        assert relerr(out[0], o["rhs"]) <= TOL
        assert np.array_equal(out[0], out[1])
