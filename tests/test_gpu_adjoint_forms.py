"""The transposed-Jacobian product over the forms of the gradient, limiter, reconstruction and flux."""
import numpy as np
import pytest

import cfd_solver_2d_gpu_amd as F
from helpers import SoaMesh
from test_gpu_adjoint import (announce, modulated_state, naca_mesh, naca_params, rel, standard_geometry_arrays,
                              wall_sets)

pytestmark = pytest.mark.gpu

FORMS = [(F.GRA_GREENGAUSS, F.LIM_BARTH, F.SOL_LLF, F.REC_LINEAR, 0),
         (F.GRA_GREENGAUSS, F.LIM_NONE, F.SOL_ROE, F.REC_CONSTANT, 0),
         (F.GRA_GREENGAUSS, F.LIM_VENKATAKRISHNAN, F.SOL_LLF, F.REC_LINEAR, 0),
         (F.GRA_LEASTSQUARE, F.LIM_NONE, F.SOL_ROE, F.REC_LINEAR, 0),
         (F.GRA_LEASTSQUARE, F.LIM_BARTH, F.SOL_ROE, F.REC_LINEAR, 0),
         (F.GRA_LEASTSQUARE, F.LIM_VENKATAKRISHNAN, F.SOL_LLF, F.REC_LINEAR, 0)]


def form_params(form, **kw):
    gradient, limiter, scheme, reconstruct, compat = form
    return naca_params(limiter=limiter, scheme=scheme, gradient=gradient, reconstruct=reconstruct,
                       compat_inv2x2=compat, **kw)


@pytest.mark.parametrize("kernels", [F.KERNELS_TILE, F.KERNELS_CELL])
@pytest.mark.parametrize("form", FORMS)
def test_vjp_forms_match_residual_differences(form, kernels):
    """Central differences with a step of 1e-7 of the state's size: truncation 1e-14 of the third
    derivative, cancellation 1e-16 / 1e-7, hence 1e-6."""
    announce(f"adjoint product vs central differences, form {form}, kernels {kernels}")
    m = naca_mesh(47, 15, 1.2)
    p = form_params(form, kernels=kernels)
    U = modulated_state(m, p)
    g = F.GPUSolver2(m, p)
    rng = np.random.default_rng(17)
    psi = rng.standard_normal(U.shape)
    g.set_state(U)
    out = g.adjoint_vjp(psi)
    v = rng.standard_normal(U.shape) * np.abs(U).mean(axis=1, keepdims=True)
    eps = 1e-7
    g.set_state(U + eps * v)
    rp = g.stage_rhs()
    g.set_state(U - eps * v)
    rm = g.stage_rhs()
    g.close()
    fd, ad = np.sum(psi * (rp - rm)) / (2 * eps), np.sum(out * v)
    assert rel(fd, ad) < 1e-6, (fd, ad)


@pytest.mark.parametrize("tile_cells", [0, 1, 37])
@pytest.mark.parametrize("form", FORMS + [(F.GRA_LEASTSQUARE, F.LIM_BARTH, F.SOL_ROE, F.REC_LINEAR, 1)])
def test_vjp_tile_and_cell_kernels_agree(form, tile_cells):
    """The two kernels add the same terms in the same order from geometry that differs by two
    roundings: a few hundred operations of 1e-16 on terms that partly cancel, hence 1e-12."""
    announce(f"adjoint product, tile vs cell kernels, form {form}, tile_cells {tile_cells}")
    m = naca_mesh(47, 15, 1.2)
    out = []
    for kw in ({"kernels": F.KERNELS_TILE, "tile_cells": tile_cells}, {"kernels": F.KERNELS_CELL}):
        p = form_params(form, **kw)
        U = modulated_state(m, p)
        g = F.GPUSolver2(m, p)
        g.set_state(U)
        out.append(g.adjoint_vjp(np.random.default_rng(23).standard_normal(U.shape)))
        g.close()
    assert np.linalg.norm(out[0] - out[1]) / np.linalg.norm(out[1]) < 1e-12


@pytest.mark.parametrize("time_advance", [F.EVO_RK3, F.EVO_EXPLICIT])
def test_adjoint_iterations_tile_and_cell_kernels_agree(time_advance):
    announce(f"adjoint iterations, tile vs cell kernels (NACA 47 x 15, 60 iterations), time advance {time_advance}")
    m = naca_mesh(47, 15, 1.2)
    out = []
    for kern in (F.KERNELS_TILE, F.KERNELS_CELL):
        p = form_params(FORMS[3], kernels=kern, cfl=0.5)
        p.time_advance = time_advance
        g = F.GPUSolver2(m, p)
        g.set_state(modulated_state(m, p))
        res, _ = g.adjoint_solve(wall_sets(m), 1.0, 60, 0.0)
        out.append((g.adjoint_state(), res.dJ_dalpha))
        g.close()
    (pt, at), (pc, ac) = out
    assert np.linalg.norm(pt - pc) / np.linalg.norm(pc) < 1e-12
    assert rel(at, ac) < 1e-11


@pytest.mark.parametrize("form", FORMS)
def test_vjp_coordinates_forms_match_differences(form):
    """Central differences over FP64 geometry with a step of 1e-7 of the local spacing: the areas of the
    thinnest cells carry 1e-16 / 1e-7 relative, ten times that where edge lengths cancel, hence 1e-5."""
    announce(f"adjoint coordinate product vs central differences, form {form}")
    m = naca_mesh(31, 9, 1.3)
    p = form_params(form)
    U = modulated_state(m, p)
    a = F.soa_arrays(m.soa)
    xy = a["node_xy"].copy()
    rng = np.random.default_rng(29)
    psi = rng.standard_normal(U.shape)
    g = F.GPUSolver2(SoaMesh(standard_geometry_arrays(a, xy)), p)
    g.set_state(U)
    _, dxy = g.adjoint_vjp(psi, coords=True)
    g.close()
    e0, e1 = a["edge_nodes"]
    L = np.hypot(xy[0][e1] - xy[0][e0], xy[1][e1] - xy[1][e0])
    hloc = np.full(xy.shape[1], np.inf)
    np.minimum.at(hloc, e0, L)
    np.minimum.at(hloc, e1, L)
    d = rng.standard_normal(xy.shape) * hloc
    eps = 1e-7
    r = []
    for s in (1, -1):
        gg = F.GPUSolver2(SoaMesh(standard_geometry_arrays(a, xy + s * eps * d)), p)
        gg.set_state(U)
        r.append(gg.stage_rhs())
        gg.close()
    fd, ad = np.sum(psi * (r[0] - r[1])) / (2 * eps), np.sum(dxy * d)
    assert rel(fd, ad) < 1e-5, (fd, ad)
