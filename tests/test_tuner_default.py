"""The tuners try what the library takes by itself, and what they return makes the handle that they timed."""
import numpy as np
import pytest

import cfd_solver_2d_gpu_amd as F
from helpers import wedge_case


@pytest.mark.parametrize("precision,threads", [(F.PREC_FP64, [256, 128, 512]), (F.PREC_MIXED, [256, 512])])
def test_candidates_hold_every_default(precision, threads):
    cand = F.autotune_candidates(precision)
    assert cand[0] == (256, 0)
    assert [th for th, cells in cand if cells == 0] == threads


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [F.PREC_FP64, F.PREC_MIXED])
@pytest.mark.parametrize("n", [64, 400])
def test_tile_shape_names_the_default(n, precision):
    """A mesh of less than one default tile per CU (8,192 cells) and one of more (320,000)."""
    print(f"[gpu-case] tile shape of the default handle, wedge {n}, precision {precision}", flush=True)
    m, p, _ = wedge_case(n, n, scheme=F.SOL_ROE)
    p.precision = precision
    g = F.GPUSolver2(m, p)
    th, cells = g.tile_shape()
    perm = g.permutation()
    g.close()
    assert th in (256, 512) and (cells < 72 if n == 64 else cells >= 150)
    for q in ((th, 0), (th, cells)):
        p.tile_threads, p.tile_cells = q
        g = F.GPUSolver2(m, p)
        assert g.tile_shape() == (th, cells) and np.array_equal(g.permutation(), perm)
        g.close()
    p.kernels = F.KERNELS_CELL
    g = F.GPUSolver2(m, p)
    assert g.tile_shape() == (0, 0)
    g.close()
