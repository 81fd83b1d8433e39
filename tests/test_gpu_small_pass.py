"""The one-pass residual and time step of small meshes against the two-pass form (the no-allocation
entry keeps it) and the oracle, over the face rules, partly filled blocks and slots, boundary faces,
a residual written over the state, whole SSP-RK3 steps, and meshes just above the limits, whose default
form is the two-pass one: those against the oracle."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from helpers import RS, random_rec, random_state, rel_l2

pytestmark = pytest.mark.gpu

TOL = 1e-13  # four fluxes of some 200 rounded operations, 2^-53 each: 9e-14
GAS = dict(Rgas=1.0, muGas=0.05, prGas=0.72, TRef=1.5, CSutherland=0.4)


def _mesh(kind):
    from dndsr_amd import bc
    from dndsr_amd import mesh as mm
    zones = dict(ymin=0, ymax=1)
    if kind == "quad1":
        return mm.periodic_quad_grid(3, 3, 1.0, 0.8), None
    if kind == "tri":
        return mm.tri_grid(7, 5, 1.0, 1.0, periodic=(True, True), jitter=0.1, seed=3), None
    if kind == "mixed":
        return mm.mixed_grid(10, 6, 1.0, 1.0, periodic=(True, False), zones=zones, jitter=0.05,
                             seed=3), [bc.BC_WALL, bc.BC_SYM]
    if kind == "tet":
        return mm.tet_grid(3, 4, 3, 1.0, 1.0, 1.0, periodic=(True, False, True), zones=zones, jitter=0.05,
                           seed=3), [bc.BC_WALL, bc.BC_WALL_INVIS]
    if kind == "quad33k":  # above both limits
        return mm.periodic_quad_grid(183, 181, 1.0, 0.8, jitter=0.1, seed=3), None
    if kind == "mixed33k":
        return mm.mixed_grid(180, 123, 1.0, 1.0, periodic=(True, False), zones=zones, jitter=0.05,
                             seed=3), [bc.BC_WALL, bc.BC_SYM]
    n = dict(tet16k=(14, 14, 14), tet33k=(18, 18, 17))[kind]  # above the viscous limit of tetrahedra, above both
    return mm.tet_grid(*n, 1.0, 1.0, 1.0, periodic=(True, False, True), zones=zones, jitter=0.05,
                       seed=3), [bc.BC_WALL, bc.BC_WALL_INVIS]


def _setup(kind, rs, viscous):
    from dndsr_amd import bc
    from dndsr_amd.cfv import VariationalReconstruction
    from dndsr_amd.euler import EulerEvaluator
    m, types = _mesh(kind)
    s = dict(maxOrder=1, intOrder=3)
    zw = {} if types is None else dict(zoneDirWeight=bc.euler_dir_weights(types, 1))
    g = VariationalReconstruction(m, dict(s, **zw)).construct()
    ev = EulerEvaluator(g, dict(riemannSolverType=rs, viscous=viscous, idealGasProperty=dict(GAS, muModel=1),
                                **(dict(bcTypes=types, bcValues=np.ones((len(types), 5))) if types else {})))
    return m, types, s, zw, g, ev


@pytest.mark.parametrize("viscous", [False, True])
@pytest.mark.parametrize("rs", ["Roe", "HLLEP"])
@pytest.mark.parametrize("kind", ["quad1", "tri", "mixed", "tet", "quad33k", "mixed33k", "tet16k", "tet33k"])
def test_same_as_two_passes(require_gpu, kind, rs, viscous):
    from dndsr_amd._lib import check, lib
    from dndsr_amd.cfv import _ptr
    print(f"\n[small pass] {kind} {rs} viscous={viscous}", flush=True)
    m, types, s, zw, g, ev = _setup(kind, rs, viscous)
    u, rec = random_state(g.nCell, 5), random_rec(g.nCell, g.M)
    du, dr, rhs, two = g.to_device(u), g.to_device(rec), g.BuildUDof(5), g.BuildUDof(5)
    dt = g.BuildUDof(1)[0]
    ev.EvaluateDt(dt, du, None, CFL=0.7)
    o = None
    if kind.endswith("k"):
        import pyoracle as po
        o = po.OracleVR(m, **s, **zw)
        if types:
            o.set_bc(types, np.ones((len(types), 5)), 1.4)
        es = po.OracleVR.euler_settings(1.4, RS[rs], 0, 1.0, 1.0, viscous=int(viscous), muModel=1, **GAS)
        dlc = o.eval_dt(es, u, 1.0, 1e100, True)[2]
    assert (g.nCell > 32768) == kind.endswith("33k") and (16384 < g.nCell <= 32768) == (kind == "tet16k")
    for r in (dr, None):
        ev.EvaluateRHS(rhs, None, du, r, r)
        if o is not None:
            want = o.eval_rhs(es, u, None if r is None else rec, dlc)
            assert rel_l2(g.to_host(rhs), want) <= 1e-12
        check(lib().dndsr_eval_rhs_noalloc(ev.ctx.h, C.byref(ev.es), _ptr(du), None if r is None else _ptr(r),
                                           _ptr(ev.deltaLambdaCell), _ptr(two)))
        ev.ctx.sync()
        a, b = g.to_host(rhs), g.to_host(two)
        # the same operations on the same values: what differs is which products are contracted
        assert rel_l2(a, b) <= TOL
        over = du.clone()  # the residual over the state it is formed from
        check(lib().dndsr_eval_rhs(ev.ctx.h, C.byref(ev.es), _ptr(over), None if r is None else _ptr(r),
                                   _ptr(ev.deltaLambdaCell), _ptr(over)))
        ev.ctx.sync()
        assert rel_l2(g.to_host(over), b) <= TOL


@pytest.mark.parametrize("kind", ["quad1", "mixed", "tet", "tet16k", "quad33k"])
def test_steps_match_oracle(require_gpu, kind):
    import pyoracle as po
    print(f"\n[small pass] steps {kind}", flush=True)
    m, types, s, zw, g, ev = _setup(kind, "HLLEP", True)
    o = po.OracleVR(m, **s, **zw)
    if types:
        o.set_bc(types, np.ones((len(types), 5)), 1.4)
    es = po.OracleVR.euler_settings(1.4, RS["HLLEP"], 0, 1.0, 1.0, viscous=1, muModel=1, **GAS)
    u = random_state(g.nCell, 5)
    du = g.to_device(u)
    dt = g.BuildUDof(1)[0]
    want = o.eval_dt(es, u, 0.3, 1e100, True)
    assert abs(ev.EvaluateDt(dt, du, None, CFL=0.3) - want[0].min()) <= 1e-13 * want[0].min()
    assert rel_l2(g.to_host(dt).ravel(), want[0].ravel()) <= 1e-13
    assert rel_l2(g.to_host(ev.deltaLambdaCell).ravel(), want[2].ravel()) <= 1e-12
    for steps, h in ((1, 0.0), (2, 0.25 * want[0].min())):  # one sweep per stage: odd and even numbers of them
        dv, dr = g.to_device(u), g.to_device(np.zeros((g.nCell, 5, g.M)))
        ev.SSPRK3(dv, dr, steps, 0.3, 1, dtFixed=h)
        uo, ro = o.ssprk3(es, u, np.zeros((g.nCell, 5, g.M)), steps, 0.3, 1, h)
        assert rel_l2(g.to_host(dv), uo) <= 1e-12 and rel_l2(g.to_host(dr), ro) <= 1e-11
