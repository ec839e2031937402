"""Caller meshes whose element_edges do not start at the side of nodes 0 and 1, or run the other way round: the
launched kernels form the centroids in the order of the element's nodes, as the caller does, so resident runs
equal single steps bit for bit there too."""
import numpy as np
import pytest

import cfd_solver_2d_gpu_amd as F
import oracle as O
from conftest import rel_l2
from helpers import SoaMesh, vortex_case, wedge_case

pytestmark = pytest.mark.gpu

ORDERS = {"0": (0, 1, 2), "1": (1, 2, 0), "2": (2, 0, 1), "back": (2, 1, 0), "swap": (1, 0, 2), "mixed": None}


def reordered(m, order):
    """The mesh with the slots (edge and neighbour) of its elements in another order; None: each its own."""
    a = {k: v.copy() for k, v in F.soa_arrays(m.soa).items()}
    n = a["element_volume"].shape[0]
    all_orders = np.array([o for o in ORDERS.values() if o])
    pick = (np.tile(order, (n, 1)) if order else all_orders[np.random.default_rng(3).integers(0, 5, n)]).T
    for key in ("element_edges", "element_neighbors"):
        a[key][:3] = np.take_along_axis(a[key][:3], pick, axis=0)
    return SoaMesh(a)


@pytest.mark.parametrize("limiter,precision", [(F.LIM_BARTH, F.PREC_FP64), (F.LIM_BARTH, F.PREC_MIXED),
                                               (F.LIM_VENKATAKRISHNAN, F.PREC_FP64)])
@pytest.mark.parametrize("order", list(ORDERS))
def test_resident_runs_equal_single_steps(order, limiter, precision):
    print(f"[gpu-case] slots in order {order}, limiter {limiter}, precision {precision}", flush=True)
    m, p, U = wedge_case(65, 33, scheme=F.SOL_ROE, limiter=limiter, precision=precision)
    a = m.arrays()["element_xy"]
    U[0] *= 1.0 + 0.05 * np.sin(3 * a[0]) * np.cos(4 * a[1])
    m = reordered(m, ORDERS[order])
    out = []
    for runs in ((9,), (1,) * 9):
        g = F.GPUSolver2(m, p)
        g.set_state(U)
        t = 0.0
        for n in runs:
            t, info = g.advance(n, t, 1e9, F.NORM_INF)
        out.append((g.get_state(), t, info.dt, np.array(info.residual[:])))
        assert g.resident_steps() == (9 if len(runs) == 1 else 0)
        g.close()
    for x, y in zip(*out):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("order", list(ORDERS))
def test_launched_steps_match_the_oracle(order):
    print(f"[gpu-case] slots in order {order}: launched steps of the periodic vortex against the oracle", flush=True)
    m, p, U = vortex_case(32)
    m = reordered(m, ORDERS[order])
    o = O.OracleSolver(m, p)
    o.set_state(U)
    g = F.GPUSolver2(m, p)
    g.set_state(U)
    t = to = 0.0
    for _ in range(3):
        t, _ = g.iteration_device(t, 1e9)
        to, _ = o.step(to, 1e9)
    assert abs(t / to - 1) < 1e-12 and rel_l2(g.get_state(), o.get_state()) < 1e-12
    g.close()
