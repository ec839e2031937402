"""Meshes in which an edge holds another edge's nodes and geometry: every edge is standard by itself, but two
elements have an edge that is not the side of their nodes.  Batches, mixed precision, fvmr_batch_advance and the tuner
serve them like other meshes."""
import numpy as np
import pytest

import cfd_solver_2d_gpu_amd as F
import oracle as O
from conftest import rel_l2
from helpers import SoaMesh, vortex_case, wedge_case
from test_gpu_resident import naca_case

pytestmark = pytest.mark.gpu


def announce(msg):
    print(f"[gpu-case] {msg}", flush=True)


def odd_mesh(m):
    """One inner edge of a 20 x 20 or larger mesh gets the nodes and geometry of another."""
    a = {k: v.copy() for k, v in F.soa_arrays(m.soa).items()}
    inner = np.flatnonzero((a["edge_elementR"] >= 0) & (a["edge_periodicPair"] < 0))
    e, f = inner[7], inner[180]
    for key in ("edge_nodes", "edge_xy", "edge_normal"):
        a[key][:, e] = a[key][:, f]
    a["edge_length"][e] = a["edge_length"][f]
    return SoaMesh(a)


def oracle_run(m, p, U, n):
    o = O.OracleSolver(m, p)
    o.set_state(U)
    t = 0.0
    for _ in range(n):
        t, _ = o.step(t, 1e9)
    return o.get_state(), t


@pytest.mark.parametrize("threads", [128, 256, 512])
@pytest.mark.parametrize("gradient", [F.GRA_GREENGAUSS, F.GRA_LEASTSQUARE])
def test_batches_match_the_oracle(gradient, threads):
    """FP64, to the 1e-12 of the tile kernels; the plain mesh beside it stays what it is without the other."""
    announce(f"a batch with a mesh whose edges are not all sides, gradient {gradient}, {threads} work-items")
    plain, p, Up = wedge_case(48, 24, scheme=F.SOL_ROE, gradient=gradient)
    m, _, _ = wedge_case(40, 20, scheme=F.SOL_ROE)
    m = odd_mesh(m)
    a = m.arrays["element_xy"]
    U = np.array(F.field_init(m, p, F.INIT_UNIFORM))
    U[0] *= 1.0 + 0.05 * np.sin(3 * a[0]) * np.cos(4 * a[1])
    p.tile_threads = threads
    b = F.BatchSolver([plain, m], [p, p])
    b.set_state(0, Up)
    b.set_state(1, U)
    t = b.advance(5, np.zeros(2), np.full(2, 1e9))
    for c, (mm, UU) in enumerate(((plain, Up), (m, U))):
        want, tw = oracle_run(mm, p, UU, 5)
        assert abs(t[c] / tw - 1) < 1e-12 and rel_l2(b.get_state(c), want) < 1e-12
    b.close()


def test_mixed_precision_keeps_the_tile_kernels():
    announce("mixed precision on a mesh whose edges are not all sides")
    m, p, U = wedge_case(40, 20, scheme=F.SOL_ROE, precision=F.PREC_MIXED)
    m = odd_mesh(m)
    U = U.copy()
    U[0] *= 1.0 + 0.05 * np.sin(3 * m.arrays["element_xy"][0])
    for kernels in (F.KERNELS_AUTO, F.KERNELS_TILE):
        p.kernels = kernels
        g = F.GPUSolver2(m, p)
        assert g.tile_shape()[0] > 0
        g.set_state(U)
        t, _ = g.advance(2, 0.0, 1e9)
        t, _ = g.advance(5, t, 1e9)
        assert g.resident_steps() == 5
        assert rel_l2(g.get_state(), oracle_run(m, p, U, 7)[0]) < 1e-6
        g.close()


def test_batch_advance_and_tuner_of_a_plain_handle():
    announce("fvmr_batch_advance and the tuner on a mesh whose edges are not all sides")
    m, p, U = vortex_case(20)
    m = odd_mesh(m)
    b = F.BatchSolver([m], [p])
    b.set_state(0, U)
    tb = b.advance(6, np.zeros(1), np.full(1, 1e9))
    g = F.GPUSolver2(m, p)
    g.set_state(U)
    t = np.zeros(1)
    F.check(F.lib().fvmr_batch_advance(g._h, 6, F._dptr(t), F._dptr(np.full(1, 1e9))), "fvmr_batch_advance")
    assert abs(t[0] / tb[0] - 1) < 1e-12 and rel_l2(g.get_state(), b.get_state(0)) < 1e-12
    g.close()
    b.close()
    th, cells, ms = F.autotune(m, p, steps=3)
    assert (th, cells) in F.autotune_candidates() and ms > 0
    p.kernels = F.KERNELS_CELL
    g = F.GPUSolver2(m, p)
    with pytest.raises(F.FvmrError):
        F.check(F.lib().fvmr_batch_advance(g._h, 1, F._dptr(t), F._dptr(t)), "fvmr_batch_advance")
    g.close()


@pytest.mark.parametrize("gradient", [F.GRA_GREENGAUSS, F.GRA_LEASTSQUARE])
def test_steady_and_adjoint_of_a_batch_of_one(gradient):
    """Against the cell kernels of a plain handle: pseudo-time iterations and the transposed product to rounding
    (1e-12; the product's terms span three orders of magnitude more than its result: 1e-9)."""
    announce(f"steady iterations and adjoint product, gradient {gradient}")
    m, p, U = naca_case(48, 21)
    p.gradient = gradient
    m = odd_mesh(m)
    psi = np.random.default_rng(5).standard_normal(U.shape)
    b = F.BatchSolver([m], [p])
    g = F.GPUSolver2(m, p)
    assert g.tile_shape() == (0, 0)
    out = []
    one = F.GPUSolver2.__new__(F.GPUSolver2)   # the one-case calls on the batch's handle
    one._h, one.n, one.mesh = b._h, U.shape[1], m
    for h in (one, g):
        h.set_state(U)
        h.steady_solve(4, 0.0)
        out.append((h.get_state(), h.adjoint_vjp(psi)))
    one._h = None
    assert np.isfinite(out[0][0]).all()
    assert rel_l2(out[0][0], out[1][0]) < 1e-12
    assert rel_l2(out[0][1], out[1][1]) < 1e-9
    b.close()
    g.close()
