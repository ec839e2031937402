"""The device order of the cells: the Hilbert walk of four bits at a time gives the order of the bitwise walk (numbering
without tiles, where the order is the walk's own), and a batch holds its cases' arrays one after the other."""
import numpy as np
import pytest

import cfd_solver_2d_gpu_amd as F
from helpers import vortex_case, wedge_case

pytestmark = pytest.mark.gpu


def bitwise(x, y, order=16):
    """Hilbert index of the integer coordinates x, y (arrays) by the textbook walk."""
    n = 1 << order
    x, y, d = x.astype(np.int64), y.astype(np.int64), np.zeros(x.shape, dtype=np.int64)
    s = n >> 1
    while s:
        rx, ry = ((x & s) > 0).astype(np.int64), ((y & s) > 0).astype(np.int64)
        d += s * s * ((3 * rx) ^ ry)
        flip = (ry == 0) & (rx == 1)
        x, y = np.where(flip, n - 1 - x, x), np.where(flip, n - 1 - y, y)
        x, y = np.where(ry == 0, y, x), np.where(ry == 0, x, y)
        s >>= 1
    return d


@pytest.mark.parametrize("case", [lambda: vortex_case(37), lambda: wedge_case(90, 41)])
def test_order_of_the_walk(case):
    print("[gpu-case] Hilbert order of the cell kernels' numbering", flush=True)
    m, p, _ = case()
    p.kernels = F.KERNELS_CELL
    g = F.GPUSolver2(m, p)
    perm = g.permutation()
    g.close()
    c = m.arrays()["element_xy"]
    lo = c.min(axis=1)
    scale = 65535 / np.max(c.max(axis=1) - lo)
    ix, iy = [np.minimum((c[k] - lo[k]) * scale, 65535).astype(np.int64) for k in range(2)]
    assert np.array_equal(perm, np.argsort(bitwise(ix, iy), kind="stable"))


def test_batch_equals_its_cases():
    print("[gpu-case] a batch of three unlike meshes against their own handles", flush=True)
    cases = [vortex_case(21), wedge_case(40, 20, scheme=F.SOL_ROE), vortex_case(34)]
    b = F.BatchSolver([c[0] for c in cases], [c[1] for c in cases])
    for k, c in enumerate(cases):
        b.set_state(k, c[2])
    t = b.advance(3, np.zeros(3), np.full(3, 1e9))
    for k, (m, p, U) in enumerate(cases):
        g = F.GPUSolver2(m, p)
        g.set_state(U)
        tk, _ = g.advance(3, 0.0, 1e9)
        assert tk == t[k] and np.array_equal(b.get_state(k), g.get_state())
        g.close()
    b.close()
