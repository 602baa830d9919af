"""GPU parity of the actuator-line path (rotor_model.c) against the FP64 oracle.

Seeded non-orthogonal box with the benchmark rotor at its centre; each stage
of the rotor_model 6 block of Flow_Solver (solvers.c:535-563) is compared with
the oracle on the same inputs.  Integer boxes must match exactly; FP64 values
within 1e-12 relative (normwise) -- the device's sqrt/asin/exp/acos may differ
from glibc's by an ulp.
"""
import importlib
import sys
from pathlib import Path

import numpy as np
import pytest

ROOT = Path(__file__).resolve().parents[1]
sys.path.insert(0, str(ROOT))
sys.path.insert(0, str(ROOT / "oracle"))
import pyoracle as po  # noqa: E402

pytestmark = pytest.mark.gpu

TOL = 1e-12


def relerr(a, b):
    a, b = np.asarray(a, dtype=np.float64), np.asarray(b, dtype=np.float64)
    d = np.linalg.norm((a - b).ravel())
    n = np.linalg.norm(b.ravel())
    return d / n if n > 0 else d


def _setup(rotor_model, deltafunc, halfwidth, nx=40, ny=36, nz=44):
    vfs = importlib.import_module("vfs-wind_amd")
    cases = importlib.import_module("vfs-wind_amd.cases")
    b = cases.box(nx, ny, nz, h=1.0, bump=0.3)
    mx, my, mz = b["da"]
    hub = (nx / 2 + 0.13, ny / 2 - 0.21, nz / 2 + 0.37)
    ts = cases.synthetic_turbine(8.0, hub, rotor_model=rotor_model, deltafunc=deltafunc, halfwidth=halfwidth,
                                 r_nacelle=1.1)
    p = vfs.make_params(mx, my, mz, per=(0, 0, 0), bctype=(10, 10, 10, 10, 5, 4), les=0)
    ctx = vfs.Context(p)
    ctx.upload("COOR", b["coor"])
    ctx.form_metrics()
    ctx.upload("UCAT", b["ucat"])
    op = po.make_params(mx, my, mz, per=(0, 0, 0), bctype=(10, 10, 10, 10, 5, 4), les=0)
    o = po.Oracle(op, b["coor"])
    o.set("ucat", b["ucat"])
    t = po.make_turbine(ts.nx, ts.ny, ts.nz, ts.xc, ts.yc, ts.zc, ts.angvel, ts.pitch, ts.r_nacelle, ts.refangle)
    alm = vfs.ALM(ctx, ts.turbine_struct(vfs), ts.nodes, ts.foils)
    return vfs, ctx, o, t, ts, alm


@pytest.mark.parametrize("rotor_model,deltafunc,halfwidth", [(6, 7, 2.0), (3, 10, 4.0), (6, 0, 4.0)],
                         ids=["model6-gauss", "model3-s4h", "model6-2h"])
def test_alm_stages(rotor_model, deltafunc, halfwidth):
    vfs, ctx, o, t, ts, alm = _setup(rotor_model, deltafunc, halfwidth)
    nb, nvb = ts.nodes.shape[:2]
    foils = po.Foils(ts.foils)
    dt = 0.05
    # airfoil_ACL at the initial positions
    cent0, _ = po.alm_elements(ts.nodes)
    tw, ch = po.alm_twist_chord(t, cent0, foils)
    assert relerr(alm.get("TWIST"), tw) <= TOL and relerr(alm.get("CHORD"), ch) <= TOL
    for step in range(2):
        # rotor_Rot
        alm.rotate(dt)
        x, u = po.alm_rotate(t, dt, ts.nodes if step == 0 else x)
        assert relerr(alm.get("NODES"), x.reshape(-1, 3)) <= TOL
        assert relerr(alm.get("NODE_VEL"), u.reshape(-1, 3)) <= TOL
        cent, dA = po.alm_elements(x)
        assert relerr(alm.get("CENT"), cent) <= TOL and relerr(alm.get("DA"), dA) <= TOL
        # Pre_process (integer boxes: exact)
        alm.preprocess()
        box = o.alm_preprocess(alm.get("CENT"))
        assert np.array_equal(alm.get("BOX").astype(np.int32), box)
        if rotor_model == 6:
            ref = po.alm_refline(t, x)
            rcent, _ = po.alm_elements(ref)
            assert relerr(alm.get("REF_CENT"), rcent) <= TOL
            rbox = o.alm_preprocess(alm.get("REF_CENT"))
            assert np.array_equal(alm.get("REF_BOX").astype(np.int32), rbox)
            scent, sbox = alm.get("REF_CENT"), rbox
        else:
            scent, sbox = alm.get("CENT"), box
        # Calc_U_lagr
        alm.u_lagr()
        ul = alm.get("U_LAGR")
        assert relerr(ul, o.alm_ulagr(scent, sbox)) <= TOL
        # Calc_F_lagr_ACL on the device's U_lagr
        alm.f_lagr()
        f, aoa, cl, cd = po.alm_flagr(t, nb, nvb, alm.get("CENT"), ul, alm.get("NODE_VEL"), alm.get("TWIST"),
                                      alm.get("CHORD"), foils)
        assert relerr(alm.get("F_LAGR"), f) <= TOL
        assert relerr(alm.get("AOA"), aoa) <= TOL
        assert relerr(alm.get("CL"), cl) <= TOL and relerr(alm.get("CD"), cd) <= TOL
        # Calc_F_eul
        alm.f_eul()
        feul = o.alm_feul(alm.get("CENT"), box, alm.get("F_LAGR"), alm.get("DA"), df=deltafunc, halfwidth=halfwidth)
        got = ctx.download("FEUL")
        assert np.abs(got).max() > 0
        assert relerr(got, feul) <= TOL
    alm.close()
    ctx.close()


def test_alm_step_matches_stages():
    vfs, ctx, o, t, ts, alm = _setup(6, 7, 2.0)
    alm.step(0.05)
    feul_step = ctx.download("FEUL")
    f_step = alm.get("F_LAGR")
    alm.close()
    alm2 = vfs.ALM(ctx, ts.turbine_struct(vfs), ts.nodes, ts.foils)
    alm2.rotate(0.05); alm2.preprocess(); alm2.u_lagr(); alm2.f_lagr(); alm2.f_eul()
    assert np.array_equal(ctx.download("FEUL"), feul_step)
    assert np.array_equal(alm2.get("F_LAGR"), f_step)
    alm2.close()
    ctx.close()


def test_alm_uref_disk():
    """Uref_ACL on the reference's own Urefdata000 disk, scaled into the box."""
    vfs, ctx, o, t, ts, alm = _setup(6, 7, 2.0)
    tb = importlib.import_module("vfs-wind_amd.turbine")
    deck = ROOT / "tests" / "golden" / "clipper_tsr5"
    # disk of radius 8 (R = 48 scaled by 6), 1R upstream of the hub
    x, tris, cent, dA = tb.read_ucd_disk(deck / "Urefdata000", 6.0, (ts.xc, ts.yc, ts.zc), (0, 0, 1), 48.0, 6.0,
                                         loc_refvel=0.5)
    alm.set_disk(cent, dA)
    uref = alm.uref()
    box = o.alm_preprocess(cent)
    u = o.alm_ulagr(cent, box)
    want = float((u[:, 2] * dA).sum() / dA.sum())
    assert abs(uref - want) <= TOL * abs(want)
    assert 0.9 < uref < 1.1  # the inflow is 1 + 5% noise
    alm.close()
    ctx.close()


CORRECTIONS = {
    "prandtl": dict(prandtl=1),
    "shen": dict(shen=1),
    "shen1": dict(shen1=1, correction_shen1=0.9),
    "lift3d": dict(correction3d_cl=1, c0_cl=1.3),
    "smooth": dict(smoothforce=2),
    "all": dict(shen=1, correction3d_cl=1, smoothforce=1),
}


@pytest.mark.parametrize("name", list(CORRECTIONS))
def test_f_lagr_corrections_and_loads(name):
    """Calc_F_lagr_ACL with each optional correction (tip-loss models, 3D lift
    correction, force smoothing; rotor_model.c:2488-2608) and Calc_forces_ACL's
    rotor sums (rotor_model.c:4148-4180) against the oracle."""
    vfs, ctx, o, t, ts, alm = _setup(6, 7, 2.0)
    alm.close()
    opts = dict(r_rotor=8.0, tsr=6.5, num_blade=ts.nodes.shape[0], **CORRECTIONS[name])
    tv = ts.turbine_struct(vfs)
    for k, v in opts.items():
        setattr(tv, k, v)
    alm = vfs.ALM(ctx, tv, ts.nodes, ts.foils)
    to = po.make_turbine(ts.nx, ts.ny, ts.nz, ts.xc, ts.yc, ts.zc, ts.angvel, ts.pitch, ts.r_nacelle, ts.refangle,
                         **opts)
    nb, nvb = ts.nodes.shape[:2]
    foils = po.Foils(ts.foils)
    alm.rotate(0.05); alm.preprocess(); alm.u_lagr(); alm.f_lagr()
    ul = alm.get("U_LAGR")
    f, aoa, cl, cd = po.alm_flagr(to, nb, nvb, alm.get("CENT"), ul, alm.get("NODE_VEL"), alm.get("TWIST"),
                                  alm.get("CHORD"), foils)
    f0 = po.alm_flagr(t, nb, nvb, alm.get("CENT"), ul, alm.get("NODE_VEL"), alm.get("TWIST"), alm.get("CHORD"), foils)[0]
    assert relerr(f, f0) > 1e-6  # the correction changes the forces
    assert relerr(alm.get("F_LAGR"), f) <= TOL
    loads = alm.loads()
    want = po.alm_loads(to, alm.get("CENT"), alm.get("F_LAGR"), ul, alm.get("DA"))
    assert np.allclose(loads, want, rtol=1e-13, atol=0)
    alm.close()
    ctx.close()


@pytest.mark.parametrize("mode", [0, 1, 2], ids=["fixed-omega", "fixed-tsr", "torque-control"])
def test_turbine_angvel_against_oracle(mode):
    """Calc_turbineangvel over three steps (the first one initialises), with
    the aerodynamic torque of vfs_alm_loads feeding the torque controller."""
    vfs, ctx, o, t, ts, alm = _setup(6, 7, 2.0)
    tc = vfs.TurbineControl(mode=mode, angvel_fixed=0.9, tsr=6.0, r_rotor=40.0, reflength_wt=5.0, refvel_wt=9.0,
                            refvel_cfd=1.0, rho_air=1.2, J_rotation=4e6, CP_max=0.45, TSR_max=7.5, X_control=2.0,
                            fixturbinegeneratortorque=0, torque_generator=0.0)
    prm = [tc.angvel_fixed, tc.tsr, tc.r_rotor, tc.reflength_wt, tc.refvel_wt, tc.refvel_cfd, tc.rho_air, tc.J_rotation,
           tc.CP_max, tc.TSR_max, tc.X_control, tc.fixturbinegeneratortorque, tc.torque_generator]
    st = np.array([ts.angvel, 0.0, 0.0, 0.0, 0.0])
    uref, dt = 0.95, 0.05
    for ti in range(3):
        w, tsr = alm.turbine_angvel(tc, dt, uref, ti, 0)
        st = po.turbine_angvel(mode, prm, dt, uref, ti, 0, st)
        assert w == pytest.approx(st[0], rel=1e-14, abs=0) and tsr == pytest.approx(st[1], rel=1e-14, abs=1e-300)
        alm.rotate(dt); alm.preprocess(); alm.u_lagr(); alm.f_lagr()
        st[2] = -alm.loads()[7]  # Torque_aero = -M_Sum
    alm.close()
    ctx.close()


@pytest.mark.parametrize("nodes_per_blade,cells,radius,off", [
    (2, (12, 9, 14), 3.0, 0.0),       # one element per blade, boxes clipped on every side
    (41, (22, 37, 70), 9.0, 6.5),     # blades that leave the box: clipped and empty boxes, a ragged union box
    (300, (30, 28, 26), 7.0, 0.0),    # more elements than one list of a brick holds
], ids=["one-element", "leaving", "897-elements"])
def test_alm_bricks_and_searches(nodes_per_blade, cells, radius, off):
    """The nearest-node search, the sampled velocity, the polar search and the
    spreading at their edges, on the oracle's chain of the same stages."""
    vfs = importlib.import_module("vfs-wind_amd")
    cases = importlib.import_module("vfs-wind_amd.cases")
    nx, ny, nz = cells
    b = cases.box(nx, ny, nz, h=1.0, bump=0.3)
    per, bc = (0, 0, 0), (10, 10, 10, 10, 5, 4)
    hub = (nx / 2 + 0.13 + off, ny / 2 - 0.21, nz / 2 + 0.37)
    ts = cases.synthetic_turbine(radius, hub, nodes_per_blade=nodes_per_blade)
    o = po.Oracle(po.make_params(*b["da"], per=per, bctype=bc, les=0), b["coor"])
    o.set("ucat", b["ucat"])
    t = po.make_turbine(ts.nx, ts.ny, ts.nz, ts.xc, ts.yc, ts.zc, ts.angvel, ts.pitch, ts.r_nacelle, ts.refangle)
    with vfs.Context(vfs.make_params(*b["da"], per=per, bctype=bc, les=0)) as ctx:
        ctx.upload("COOR", b["coor"])
        ctx.form_metrics()
        ctx.upload("UCAT", b["ucat"])
        alm = vfs.ALM(ctx, ts.turbine_struct(vfs), ts.nodes, ts.foils)
        try:
            alm.step(0.03)
            box, rbox = o.alm_preprocess(alm.get("CENT")), o.alm_preprocess(alm.get("REF_CENT"))
            assert np.array_equal(alm.get("BOX").astype(np.int32), box)
            assert np.array_equal(alm.get("REF_BOX").astype(np.int32), rbox)
            ul = alm.get("U_LAGR")
            assert relerr(ul, o.alm_ulagr(alm.get("REF_CENT"), rbox)) <= TOL
            f, aoa, cl, cd = po.alm_flagr(t, *ts.nodes.shape[:2], alm.get("CENT"), ul, alm.get("NODE_VEL"), alm.get("TWIST"),
                                          alm.get("CHORD"), po.Foils(ts.foils))
            assert relerr(alm.get("CL"), cl) <= TOL and relerr(alm.get("F_LAGR"), f) <= TOL
            want = o.alm_feul(alm.get("CENT"), box, alm.get("F_LAGR"), alm.get("DA"), df=7, halfwidth=2.0)
            assert np.abs(want).max() > 0
            assert relerr(ctx.download("FEUL"), want) <= TOL
        finally:
            alm.close()
