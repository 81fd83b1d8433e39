"""The implicit loop's LU-SGS solves, scalar and Roe-Jacobian block, against the oracle where their layout
changes form: 3, 4 and 6 faces per cell, mixed cells with an absent slot, boundary faces, colours
smaller than a wavefront, two colours and more (half sums), Gauss-Seidel (in place) and Jacobi (two
arrays), one and several symmetric sweeps, FP64 and FP32."""
from __future__ import annotations

import numpy as np
import pytest

from helpers import RS, colour_scan_order, random_state, rel_l2

pytestmark = pytest.mark.gpu


def _mesh(kind):
    from dndsr_amd import bc
    from dndsr_amd import mesh as mm
    if kind == "tri":
        return mm.tri_grid(9, 7, 1.0, 1.0, periodic=(True, True), jitter=0.1, seed=3), None
    if kind == "mixed":
        return mm.mixed_grid(10, 6, 1.0, 1.0, periodic=(True, True), jitter=0.05, seed=3), None
    if kind == "bounded":
        return mm.mixed_grid(10, 6, 1.0, 1.0, periodic=(True, False), zones=dict(ymin=0, ymax=1), jitter=0.05,
                             seed=3), [bc.BC_WALL, bc.BC_SYM]
    if kind == "tet":
        return mm.tet_grid(4, 5, 3, 1.0, 1.0, 1.0, periodic=(True,) * 3, jitter=0.05, seed=3), None
    return mm.periodic_hex_grid(7, 5, 3, 1.0, 1.0, 1.0, jitter=0.1, seed=3), None


@pytest.mark.parametrize("block", [False, True], ids=["scalar", "block"])
@pytest.mark.parametrize("kind", ["tri", "mixed", "bounded", "tet", "hex"])
@pytest.mark.parametrize("gs,sgsIter", [(1, 0), (1, 3), (0, 2)])
def test_one_iteration_matches_oracle(require_gpu, kind, gs, sgsIter, block):
    import pyoracle as po
    from dndsr_amd import bc
    from dndsr_amd.cfv import VariationalReconstruction
    from dndsr_amd.euler import EulerEvaluator
    print(f"\n[sgs solve] {kind} gs={gs} sgsIter={sgsIter} block={block}", flush=True)
    m, types = _mesh(kind)
    s = dict(maxOrder=1, intOrder=3)
    if types:
        s["zoneDirWeight"] = bc.euler_dir_weights(types, 1)
    o = po.OracleVR(m, **s)
    g = VariationalReconstruction(m, s).construct()
    vals = None if types is None else np.ones((len(types), 5))
    if types:
        o.set_bc(types, vals, 1.4)
    ev = EulerEvaluator(g, dict(riemannSolverType="Roe", useRoeJacobian=block,
                                **(dict(bcTypes=types, bcValues=vals) if types else {})))
    es = po.OracleVR.euler_settings(1.4, RS["Roe"], useRoeJacobian=int(block))
    assert (g.colors().max() >= 2) == (kind != "tri")  # three colours: inner ones keep half sums
    u0 = random_state(g.nCell, 5)
    kw = dict(CFL=5.0, sgsIter=sgsIter, maxIter=1, minIter=1, tol=0.0)
    uo, *_ = o.implicit_euler_step(es, u0, np.zeros((o.nCell, 5, o.M)), 0.2, gsUpdate=gs,
                                   scanOrder=colour_scan_order(g.colors()), **kw)
    for fp32 in (False, True):
        du, dr = g.to_device(u0), g.BuildURec(5)
        ev.ImplicitEulerStep(du, dr, 0.2, jacobiCode=gs, fp32Sweeps=fp32, **kw)
        # FP64: rounding (blocks: times the condition of their inverses); FP32: 2 (1 + sgsIter) sweeps
        # of sums of K terms (blocks: 5 K) rounded at 2^-24 each, relative to the increment (about
        # 1e-1 of the state here)
        d = rel_l2(g.to_host(du) - u0, uo - u0)
        assert d <= (2e-6 if fp32 else 1e-11 if block else 1e-12), (fp32, d)
        print(f"[sgs solve] fp32={fp32} {d:.2e}", flush=True)
    assert rel_l2(uo, u0) > 1e-3
