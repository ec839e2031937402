"""The transposed-Jacobian product over the forms of the gradient, limiter, reconstruction and flux."""
import numpy as np
import pytest

import cfd_solver_2d_gpu_amd as F
from test_gpu_adjoint import announce, modulated_state, naca_mesh, naca_params, rel

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
