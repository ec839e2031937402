"""The tiles that the library groups a Hilbert order into, over the device order that a handle reports: on the
GPU, fields are bit for bit those of the caller's order, whatever the mesh's cells look like."""
import numpy as np
import pytest

import cfd_solver_2d_gpu_amd as F
from helpers import SoaMesh, vortex_case, wedge_case


def ogrid_case(ni=96, nj=60):
    """Cells up to 40 times longer than wide at the wall."""
    m = F.Mesh.generate(F.GEN_CYLINDER_OGRID, ni, nj, a=0.5, b=20.0, c=1.12)
    inf = list(F.ruvp_from_mach(0.4, 3.0))
    p = F.default_params(inf_ruvp=inf, inlet_ruvp=inf, outlet_ruvp=inf, CFL=0.5, time_advance=F.EVO_RK3)
    U = F.field_init(m, p)
    a = m.arrays()["element_xy"]
    U[0] *= 1.0 + 0.01 * np.sin(a[0]) * np.cos(a[1])
    return m, p, U


CASES = {"ogrid": ogrid_case, "vortex": lambda: vortex_case(37), "wedge": lambda: wedge_case(70, 41, scheme=F.SOL_ROE)}


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [F.PREC_FP64, F.PREC_MIXED])
@pytest.mark.parametrize("tile_cells", [0, 1, 40, 200, 400])
@pytest.mark.parametrize("case", list(CASES))
def test_grouped_tiles_give_the_same_fields(case, tile_cells, precision):
    print(f"[gpu-case] grouped tiles: {case}, tile_cells {tile_cells}, precision {precision}", flush=True)
    m, p, U = CASES[case]()
    p.precision, p.tile_cells, p.kernels = precision, tile_cells, F.KERNELS_TILE
    out = []
    for renumber in (F.RENUMBER_HILBERT, F.RENUMBER_NONE):
        p.renumber = renumber
        g = F.GPUSolver2(m, p)
        assert np.array_equal(np.sort(g.permutation()), np.arange(m.num_element))
        g.set_state(U)
        t, info = g.advance(3, 0.0, 1e9, F.NORM_INF)   # the launched kernels
        t, info = g.advance(5, t, 1e9, F.NORM_INF)     # the resident kernel where it fits
        out.append((g.get_state(), t, info.dt, np.array(info.residual[:])))
        g.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("kernels", [F.KERNELS_AUTO, F.KERNELS_TILE])
def test_edges_that_are_not_sides_use_the_cell_kernels(kernels):
    """An edge that holds another edge's nodes and geometry: every edge is still standard by itself, but two
    elements have a side that does not join their nodes, so the tiles cannot form it from them."""
    print(f"[gpu-case] an edge that is no side of its elements, kernels {kernels}", flush=True)
    m, p, U = vortex_case(20)
    a = {k: v.copy() for k, v in F.soa_arrays(m.soa).items()}
    inner = np.flatnonzero((a["edge_elementR"] >= 0) & (a["edge_periodicPair"] < 0))
    e, f = inner[7], inner[180]
    for key in ("edge_nodes", "edge_xy", "edge_normal"):
        a[key][:, e] = a[key][:, f]
    a["edge_length"][e] = a["edge_length"][f]
    out = []
    for kern in (kernels, F.KERNELS_CELL):
        p.kernels = kern
        g = F.GPUSolver2(SoaMesh(a), p)
        g.set_state(U)
        g.advance(5, 0.0, 1e9)
        out.append(g.get_state())
        g.close()
    assert np.array_equal(*out)
