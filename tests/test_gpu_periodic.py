"""Contra2Cart's periodic ghosts formed in the interior pass, boundary rules of
ghosts that stand for another point, the pressure update that writes its own
periodic copies: every combination of periodic directions and walls against the
oracle, ghosts included."""
import importlib

import numpy as np
import pytest

import pyoracle as po
from helpers import cases, relerr, vfs

pytestmark = pytest.mark.gpu

TOL = 1e-12  # relative to the field's maximum: sums of tens of rounded terms
# bctype per periodicity: no-slip, slip, and walls on two axes (the snapshot path)
BCS = {(1, 1): (100, 100, 1, 10, 100, 100), (1, 0): (100, 100, 1, 1, 1, 10), (0, 1): (10, 1, 10, 1, 100, 100),
       (0, 0): (1, 10, 1, 1, 10, 1)}


@pytest.mark.parametrize("blanked", [False, True])
@pytest.mark.parametrize("per", list(BCS), ids=str)
@pytest.mark.parametrize("cells", [(4, 4, 5), (18, 7, 12)], ids=str)
def test_periodic_combinations(cells, per, blanked):
    c = cases.channel(*cells)
    kw = dict(per=(per[0], 0, per[1]), bctype=BCS[per], ren=c.ren, dt=1e-3, inlet_flux=c.inlet_flux)
    o = po.Oracle(po.make_params(*c.da, **kw), c.coor)
    rng = np.random.default_rng(5)
    fields = {"ucont": c.ucont + 1e-3 * rng.standard_normal(c.ucont.shape), "p": rng.standard_normal(o.shape),
              "ucat_old": rng.standard_normal(c.ucont.shape)}
    for f, v in fields.items():
        o.set(f, v)
    with vfs.Context(vfs.make_params(*c.da, **kw)) as ctx:
        ctx.upload("COOR", c.coor)
        ctx.form_metrics()
        if blanked:
            nv = np.zeros(o.shape)
            nv[2, 2, 2:4] = 1.0  # (off the periodic planes, whose nvert copies the host fills)
            o.m["nvert"][...] = nv
            ctx.upload("NVERT", nv)
        for f, v in fields.items():
            ctx.upload(f.upper(), v)
        for run in ("contra2cart", "eddy_viscosity", "calc_k_flux", "pressure_gradient", "formfunction2", "runge_kutta",
                    "poisson_rhs"):
            if run == "runge_kutta" and (per != (1, 1) or blanked):
                continue  # (the stages take Contra2Cart as idempotent, which it is not on such boxes)
            if run == "calc_k_flux":
                o.mean_k_area(), ctx.mean_k_area()
            getattr(o, run)()
            getattr(ctx, run)()
        phi = rng.standard_normal(o.shape)
        o.set("phi", phi)
        ctx.upload("PHI", phi)
        for run in ("update_pressure", "projection"):
            getattr(o, run)()
            getattr(ctx, run)()
        for f in ("ucat", "nu_t", "rhs", "ucont", "b", "phi", "p"):
            assert relerr(ctx.download(f.upper()), o[f]) <= TOL, f
        assert abs(ctx.divergence() - o.divergence()) <= TOL * max(1.0, abs(o.divergence()))
