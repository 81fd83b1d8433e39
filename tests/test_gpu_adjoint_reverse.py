"""The reverse-mode fluxes behind the residual's vector-Jacobian product for the flux forms that
test_gpu_adjoint.py does not name (every Roe eigenvalue scheme, its batched forms, the second HLLE+
form), subsonic and with supersonic faces, on a linear mesh (face kernel, three points on two
wavefronts) and a quadratic one (point kernel): against central differences of the device residual."""
from __future__ import annotations

import pytest

from helpers import random_rec, random_state, small_mesh

pytestmark = pytest.mark.gpu

FORMS = [(f"Roe_M{k}", b) for k in range(1, 9) for b in (0, 1) if not (b and k > 5)] + [("HLLEP_V1", 0)]


@pytest.mark.parametrize("rs,batch", FORMS, ids=[f"{r}{'b' if b else ''}" for r, b in FORMS])
@pytest.mark.parametrize("kind,order,mach", [("2d", 1, 0.3), ("3d", 2, 1.0)])
def test_vjp_matches_central_differences(require_gpu, kind, order, mach, rs, batch):
    import torch
    from dndsr_amd import adjoint
    from dndsr_amd.cfv import VariationalReconstruction
    from dndsr_amd.euler import EulerEvaluator
    print(f"\n[adjoint reverse] {kind} p{order} {rs} batch={batch}", flush=True)
    g = VariationalReconstruction(small_mesh(kind, jitter=0.1), dict(maxOrder=order, intOrder=5)).construct()
    ev = EulerEvaluator(g, dict(riemannSolverType=rs, rsMeanValueEig=batch))
    s = random_state(g.nCell, 5)
    s[:, 4] -= 0.5 * (s[:, 1:4] ** 2).sum(1) / s[:, 0]
    s[:, 1:4] *= mach / 0.3
    s[:, 4] += 0.5 * (s[:, 1:4] ** 2).sum(1) / s[:, 0]
    u, rec = g.to_device(s), g.to_device(random_rec(g.nCell, g.M, 5, seed=6, amp=2e-2))
    ev.EvaluateDt(torch.zeros_like(u[0]), u, None, 1.0)
    dlc = ev.deltaLambdaCell.clone()
    gen = torch.Generator(device="cpu").manual_seed(3)
    rnd = lambda t, a: torch.randn(t.shape, generator=gen, dtype=torch.float64).to(t.device) * a  # noqa: E731
    lam, vu, vr = rnd(u, 1.0), rnd(u, 1e-1), rnd(rec, 1e-2)
    uBar, recBar = adjoint.rhs_vjp(ev, u, rec, dlc, lam)
    lhs = float((uBar * vu).sum() + (recBar * vr).sum())
    eps = 1e-6
    d = adjoint._eval_rhs(ev, u + eps * vu, rec + eps * vr, dlc) - adjoint._eval_rhs(ev, u - eps * vu, rec - eps * vr,
                                                                                     dlc)
    fd = float((lam * d).sum()) / (2 * eps)
    # central differences of piecewise smooth fluxes: rounding 1e-16 / eps and the kinks a step crosses
    assert abs(lhs - fd) <= 1e-6 * max(abs(fd), float((uBar * vu).abs().sum()) * 1e-2), (lhs, fd)
