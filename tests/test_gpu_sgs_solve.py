"""The implicit loop's LU-SGS solve against the oracle where its layout changes form: 3, 4 and 6
faces per cell, mixed cells with an absent slot, colours smaller than a wavefront, Gauss-Seidel
(in place) and Jacobi (two arrays), one and several symmetric sweeps, FP64 and FP32."""
from __future__ import annotations

import numpy as np
import pytest

from helpers import RS, colour_scan_order, random_state, rel_l2

pytestmark = pytest.mark.gpu


def _mesh(kind):
    from dndsr_amd import mesh as mm
    if kind == "tri":
        return mm.tri_grid(9, 7, 1.0, 1.0, periodic=(True, True), jitter=0.1, seed=3)
    if kind == "mixed":
        return mm.mixed_grid(10, 6, 1.0, 1.0, periodic=(True, True), jitter=0.05, seed=3)
    if kind == "tet":
        return mm.tet_grid(4, 5, 3, 1.0, 1.0, 1.0, periodic=(True,) * 3, jitter=0.05, seed=3)
    return mm.periodic_hex_grid(7, 5, 3, 1.0, 1.0, 1.0, jitter=0.1, seed=3)


@pytest.mark.parametrize("kind", ["tri", "mixed", "tet", "hex"])
@pytest.mark.parametrize("gs,sgsIter", [(1, 0), (1, 3), (0, 2)])
def test_one_iteration_matches_oracle(require_gpu, kind, gs, sgsIter):
    import pyoracle as po
    from dndsr_amd.cfv import VariationalReconstruction
    from dndsr_amd.euler import EulerEvaluator
    print(f"\n[sgs solve] {kind} gs={gs} sgsIter={sgsIter}", flush=True)
    m = _mesh(kind)
    s = dict(maxOrder=1, intOrder=3)
    o = po.OracleVR(m, **s)
    g = VariationalReconstruction(m, s).construct()
    ev = EulerEvaluator(g, dict(riemannSolverType="Roe"))
    es = po.OracleVR.euler_settings(1.4, RS["Roe"])
    u0 = random_state(g.nCell, 5)
    kw = dict(CFL=5.0, sgsIter=sgsIter, maxIter=1, minIter=1, tol=0.0)
    uo, *_ = o.implicit_euler_step(es, u0, np.zeros((o.nCell, 5, o.M)), 0.2, gsUpdate=gs,
                                   scanOrder=colour_scan_order(g.colors()), **kw)
    for fp32 in (False, True):
        du, dr = g.to_device(u0), g.BuildURec(5)
        ev.ImplicitEulerStep(du, dr, 0.2, jacobiCode=gs, fp32Sweeps=fp32, **kw)
        # FP64: rounding; FP32: 2 (1 + sgsIter) sweeps of sums of K terms rounded at 2^-24
        # each, relative to the increment (about 1e-1 of the state here)
        d = rel_l2(g.to_host(du) - u0, uo - u0)
        assert d <= (2e-6 if fp32 else 1e-12), (fp32, d)
    assert rel_l2(uo, u0) > 1e-3
