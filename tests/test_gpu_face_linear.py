"""The linear residual kernels (maxOrder 1 or no reconstruction) against the oracle on every face rule
they take, odd face counts, periodic shifts, boundary faces left to their own passes, viscous or not, and
flux forms that read deltaLambdaCell or share the face's eigenvalues.  The meshes are small, so the
default entry runs the one-pass kernel (the face kernel on hexahedra); the no-allocation entry, always
face kernel and gather, is compared with the oracle as well.  Then the rounding of both forms."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from helpers import RS, random_rec, random_state, rel_l2

pytestmark = pytest.mark.gpu

GAS = dict(Rgas=1.0, muGas=0.05, prGas=0.72, TRef=1.5, CSutherland=0.4)


def _mesh(kind):
    from dndsr_amd import bc
    from dndsr_amd import mesh as mm
    if kind == "tri":
        return mm.tri_grid(7, 5, 1.0, 1.0, periodic=(True, True), jitter=0.1, seed=3), None
    if kind == "quad":
        return mm.periodic_quad_grid(9, 7, 1.0, 0.8, jitter=0.1, seed=3), None
    if kind == "mixed":
        return mm.mixed_grid(10, 6, 1.0, 1.0, periodic=(True, False), zones=dict(ymin=0, ymax=1), jitter=0.05,
                             seed=3), [bc.BC_WALL, bc.BC_SYM]
    if kind == "hex":
        return mm.periodic_hex_grid(5, 4, 3, 1.0, 1.0, 1.0, jitter=0.1, seed=3), None
    return mm.tet_grid(3, 4, 3, 1.0, 1.0, 1.0, periodic=(True, False, True), zones=dict(ymin=0, ymax=1),
                       jitter=0.05, seed=3), [bc.BC_WALL, bc.BC_WALL_INVIS]


@pytest.mark.parametrize("kind,intOrder", [("tri", 3), ("quad", 3), ("quad", 5), ("mixed", 3), ("hex", 3),
                                           ("tet", 3), ("tet", 4)])
@pytest.mark.parametrize("rs,batch", [("Roe", 0), ("HLLEP", 0), ("Roe_M1", 1)])
def test_residual_matches_oracle(require_gpu, kind, intOrder, rs, batch):
    import pyoracle as po
    from dndsr_amd import bc
    from dndsr_amd._lib import check, lib
    from dndsr_amd.cfv import VariationalReconstruction, _ptr
    from dndsr_amd.euler import EulerEvaluator
    print(f"\n[face linear] {kind} intOrder {intOrder} {rs} batch={batch}", flush=True)
    m, types = _mesh(kind)
    s = dict(maxOrder=1, intOrder=intOrder)
    zw = {} if types is None else dict(zoneDirWeight=bc.euler_dir_weights(types, 1))
    o = po.OracleVR(m, **s, **zw)
    g = VariationalReconstruction(m, dict(s, **zw)).construct()
    if types:
        o.set_bc(types, np.ones((len(types), 5)), 1.4)
    u, rec = random_state(g.nCell, 5), random_rec(g.nCell, g.M)
    du, dr, rhs = g.to_device(u), g.to_device(rec), g.BuildUDof(5)
    for viscous in (False, True):
        es = po.OracleVR.euler_settings(1.4, RS[rs], batch, 1.0, 1.0, viscous=int(viscous), muModel=1, **GAS)
        ev = EulerEvaluator(g, dict(riemannSolverType=rs, rsMeanValueEig=batch, viscous=viscous,
                                    idealGasProperty=dict(GAS, muModel=1),
                                    **(dict(bcTypes=types, bcValues=np.ones((len(types), 5))) if types else {})))
        ev.EvaluateDt(g.BuildUDof(1)[0], du, None, CFL=1.0)
        dlc = o.eval_dt(es, u, 1.0, 1e100, True)[2]
        for r, d in ((rec, dr), (None, None)):
            ev.EvaluateRHS(rhs, None, du, d, d)
            want, two = o.eval_rhs(es, u, r, dlc), g.BuildUDof(5)
            assert rel_l2(g.to_host(rhs), want) <= 1e-12, (viscous, r is None)
            check(lib().dndsr_eval_rhs_noalloc(ev.ctx.h, C.byref(ev.es), _ptr(du), _ptr(d),
                                               _ptr(ev.deltaLambdaCell), _ptr(two)))
            ev.ctx.sync()
            assert rel_l2(g.to_host(two), want) <= 1e-12, (viscous, r is None)


@pytest.mark.parametrize("kind", ["quad", "tri", "tet"])
def test_rounding_of_a_linear_pressure_field(require_gpu, kind):
    """Fluid at rest with a linear pressure: the momentum residual is -1/V sum s w n (p_L + p_R) / 2, formed
    here in extended precision from the same metrics and coefficients.  A rounding is uniform in half a
    unit of the last place: 0.408 2^-53 of the value (rms over its mantissa).  Per point of pA / G the states of
    both sides, their pressure, and the products with n and w are rounded (3 in the mean of the two), per
    face the G - 1 partial sums of k pA / G, per cell the K - 1 sums of its faces; a rounding that all points of a face
    share would weigh sqrt(G) times as much.  Margin 1.1 for the spread of areas."""
    from dndsr_amd import mesh as mm
    from dndsr_amd._lib import check, lib
    from dndsr_amd.cfv import VariationalReconstruction, _ptr
    from dndsr_amd.euler import EulerEvaluator
    print(f"\n[face linear] rounding {kind}", flush=True)
    LD, per = np.longdouble, (True,) * 3
    m = {"quad": lambda: mm.periodic_quad_grid(40, 40, 1.0, 1.0, jitter=0.1, seed=3),
         "tri": lambda: mm.tri_grid(40, 40, 1.0, 1.0, periodic=(True, True), jitter=0.1, seed=3),
         "tet": lambda: mm.tet_grid(9, 9, 9, 1.0, 1.0, 1.0, periodic=per, jitter=0.05, seed=3)}[kind]()
    g = VariationalReconstruction(m, dict(maxOrder=1, intOrder=3)).construct()
    c, f = g.cell_metrics(), g.face_metrics()
    ev = EulerEvaluator(g, dict(riemannSolverType="Roe"))
    slope, M, N = np.array([0.02, -0.03, 0.015][:m.dim]), g.M, g.nCell
    bary, sc = c["cent"][:, :m.dim] + c["scale"][:, None] * c["moment"], c["scale"]
    u, rec = np.zeros((N, 5)), np.zeros((N, 5, M))
    u[:, 0], u[:, 4] = 1.0, 2.5 + (bary - 0.5) @ slope
    rec[:, 4] = slope * sc[:, None]
    du, dr, rhs, two = g.to_device(u), g.to_device(rec), g.BuildUDof(5), g.BuildUDof(5)
    ev.EvaluateDt(g.BuildUDof(1)[0], du, None, CFL=1.0)
    ev.EvaluateRHS(rhs, None, du, dr, dr)
    check(lib().dndsr_eval_rhs_noalloc(ev.ctx.h, C.byref(ev.es), _ptr(du), _ptr(dr), _ptr(ev.deltaLambdaCell),
                                       _ptr(two)))
    ev.ctx.sync()
    cL, cR = m.face2cell.T
    p = LD(0)
    for q in range(g.nGFace):
        x = f["pts"][:, q, :m.dim].astype(LD)
        sides = []
        for cell, sh in ((cL, 0), (cR, m.faceShift[:, :m.dim].astype(LD))):
            d = (x + sh - c["cent"][cell][:, :m.dim]) / sc[cell].astype(LD)[:, None] - c["moment"][cell]
            sides.append(u[cell, 4].astype(LD) + (d * rec[cell, 4]).sum(1))
        pm = (LD(1.4) - 1) * (sides[0] + sides[1]) / 2
        p = p + (pm * f["wJDet"][:, q])[:, None] * f["norms"][:, q].astype(LD)
    want = np.zeros((N, 3), LD)
    np.add.at(want, cL, -p)
    np.add.at(want, cR, p)
    want /= c["vol"].astype(LD)[:, None]
    K, G, d = np.diff(m.cell2facePtr).max(), g.nGFace, m.dim
    A = np.add.reduceat(f["area"][m.cell2face], m.cell2facePtr[:-1]) / K
    unit = 0.408 * 2.0 ** -53 * np.sqrt(np.mean((A / c["vol"]) ** 2))  # p = 1
    bound = 1.1 * unit * np.sqrt(K / d * (3 / G + sum((k / G) ** 2 for k in range(2, G + 1))) + (K - 1) / d)
    for out in (rhs, two):
        e = (g.to_host(out)[:, 1:1 + d] - want[:, :d]).astype(float)
        assert np.sqrt(np.mean(e ** 2)) <= bound, np.sqrt(np.mean(e ** 2)) / bound
