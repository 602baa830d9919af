"""The k-marching passes choose the planes per block by the grid: runs of one
plane on small grids, runs that do not divide the plane count and long runs,
against the oracle."""
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
