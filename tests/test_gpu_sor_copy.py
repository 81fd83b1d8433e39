"""The SOR sweep's matrices: a copy of A^-1 B in the order of the sweep's cell lists, made at
construction (SORInstead) or by the second sweep, and A^-1 B in cell order for the first one and those
captured before there is a copy; replacing the coefficients refreshes the copy, also for a captured sweep.  Odd
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


def _hex(order=3):
    from dndsr_amd import mesh as mm
    o, g, _ = _pair(mm.periodic_hex_grid(7, 5, 5, 1.0, 1.0, 1.0, jitter=0.1, seed=2), order, relax=0.9)
    return g, g.to_device(random_state(g.nCell, 3)), g.to_device(random_rec(g.nCell, g.M))


@pytest.mark.parametrize("atConstruct", [False, True])
def test_copy_is_made_once(require_gpu, atConstruct):
    import torch
    from dndsr_amd import mesh as mm
    print(f"\n[sor copy] memory, at construction {atConstruct}", flush=True)
    keep = _hex()
    keep[0].DoReconstructionSOR(keep[2], keep[1])  # kernels loaded
    m = mm.periodic_hex_grid(13, 11, 9, 1.0, 1.0, 1.0, jitter=0.1, seed=2)
    _, g, _ = _pair(m, 3, relax=0.9, sor=atConstruct)
    du, dr = g.to_device(random_state(g.nCell, 3)), g.to_device(random_rec(g.nCell, g.M))
    free = []
    for _ in range(4):
        torch.cuda.synchronize()
        free.append(torch.cuda.mem_get_info()[0])
        g.DoReconstructionSOR(dr, du)
    assert free[0] == free[1] and (free[1] == free[2]) == atConstruct and free[2] == free[3], free


def test_sweeps_on_several_streams(require_gpu):
    import torch
    print("\n[sor copy] streams", flush=True)
    g, du, dr = _hex()
    other, _, _ = _hex()
    want = dr.clone()
    other.DoReconstructionSOR(want, du)
    x = torch.randn(4096, 4096, device=du.device)
    fields = [dr.clone() for _ in range(3)]
    streams = [torch.cuda.Stream() for _ in range(3)]
    torch.cuda.synchronize()
    for s, r in zip(streams, fields):
        with torch.cuda.stream(s):
            for _ in range(8):  # the stream's work before the sweep: the next stream's is issued meanwhile
                x @ x
            g.DoReconstructionSOR(r, du)
    torch.cuda.synchronize()
    for r in fields:
        assert torch.equal(r, want)


@pytest.mark.parametrize("sweptBefore", [False, True])
def test_captured_sweep_reads_new_coefficients(require_gpu, sweptBefore):
    import torch
    print(f"\n[sor copy] capture, swept before {sweptBefore}", flush=True)
    g, du, dr = _hex()
    A, b = g.get_matrixAAInvB()
    for _ in range(2 * sweptBefore):
        g.DoReconstructionSOR(dr.clone(), du)
    r, graph = dr.clone(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        g.DoReconstructionSOR(r, du)
    for scale in (1.0, 0.5, 0.25):
        g.set_matrixAAInvB(scale * A, scale * b)
        want = dr.clone()
        g.DoReconstructionSOR(want, du)
        r.copy_(dr)
        graph.replay()
        torch.cuda.synchronize()
        # caller's order or list order: the same operations on the same values
        assert torch.equal(r, want), scale
