"""The SOR sweep's two matrix sources: a context's first sweep reads A^-1 B in cell order, later ones a
copy in the order of the sweep's cell lists; replacing the coefficients refreshes the copy.  Odd
periodic sizes (colours of a few cells beside the large ones) and a bounded mesh (cells with and
without a boundary face); every sweep against the oracle's SOR in colour order."""
from __future__ import annotations

import pytest

from helpers import colour_scan_order, random_rec, random_state, rel_l2
from test_gpu_sor import _bounded, _pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,order", [("hex", 2), ("hex", 3), ("tri", 3), ("box", 1)])
def test_later_sweeps_and_new_coefficients(require_gpu, kind, order):
    import torch
    from dndsr_amd import mesh as mm
    print(f"\n[sor copy] {kind} p{order}", flush=True)
    if kind == "box":
        args = (*_bounded("3d"),)
        m, extra = args[0], args[1:]
    else:
        m = (mm.periodic_hex_grid(7, 5, 5, 1.0, 1.0, 1.0, jitter=0.1, seed=2) if kind == "hex"
             else mm.tri_grid(7, 5, 1.0, 1.0, periodic=(True, True), jitter=0.1, seed=2))
        extra = ()
    o, g, ev = _pair(m, order, *extra, relax=0.9)
    scan = colour_scan_order(g.colors())
    A, b = o.vr_coeffs()
    u, rec = random_state(g.nCell, 3), random_rec(g.nCell, g.M)
    g.set_matrixAAInvB(A, b)
    du, dr = g.to_device(u), g.to_device(rec)
    for sweep in range(3):
        g.DoReconstructionSOR(dr, du)
        rec = o.vr_sor(rec, u, scan)
        assert rel_l2(g.to_host(dr), rec) <= 1e-12, sweep
    g.set_matrixAAInvB(0.5 * A, 0.5 * b)  # the copy of the old ones must go
    other = _pair(m, order, *extra, relax=0.9)
    other[1].set_matrixAAInvB(0.5 * A, 0.5 * b)
    r1, r2 = dr.clone(), dr.clone()
    g.DoReconstructionSOR(r1, du)
    other[1].DoReconstructionSOR(r2, du)  # that context's first sweep: no copy
    assert torch.equal(r1, r2) and not torch.equal(r1, dr)
