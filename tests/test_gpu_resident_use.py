"""Which runs the resident kernel serves: where it is meant to, it must be the one that has run, so that the
comparisons with the launched kernels compare the two."""
import numpy as np
import pytest

import cfd_solver_2d_gpu_amd as F
from helpers import wedge_case
from test_gpu_resident import CASES, naca_case

pytestmark = pytest.mark.gpu


def announce(msg):
    print(f"[gpu-case] {msg}", flush=True)


@pytest.mark.parametrize("precision", [F.PREC_FP64, F.PREC_MIXED])
@pytest.mark.parametrize("case", list(CASES))
def test_runs_of_small_meshes_are_resident(case, precision, golden_dir):
    """Runs of 4 steps and more; not mixed precision with periodic faces (the vortex)."""
    announce(f"resident steps of a run: {case}, precision {precision}")
    m, p, U = CASES[case](golden_dir)
    p.precision = precision
    served = not (precision == F.PREC_MIXED and case.startswith("vortex"))
    g = F.GPUSolver2(m, p)
    g.set_state(U)
    t, _ = g.advance(3, 0.0, 1e9)
    assert g.resident_steps() == 0
    t, _ = g.advance(4, t, 1e9)
    t, _ = g.advance(9, t, 1e9)
    assert g.resident_steps() == (13 if served else 0)
    g.use_resident(False)
    g.advance(9, t, 1e9)
    assert g.resident_steps() == (13 if served else 0)
    g.close()


@pytest.mark.parametrize("tile_cells,served", [(61, True), (1, False)])
def test_tile_counts(tile_cells, served):
    announce(f"resident steps with tiles of {tile_cells} cells")
    m, p, U = wedge_case(45, 22, scheme=F.SOL_ROE)   # 1,980 cells: 33 tiles, and more than the device holds
    p.tile_cells = tile_cells
    g = F.GPUSolver2(m, p)
    g.set_state(U)
    g.advance(7, 0.0, 1e9)
    assert g.resident_steps() == (7 if served else 0)
    g.close()


def test_pseudo_time_iterations_are_resident():
    announce("resident pseudo-time iterations")
    m, p, U = naca_case(48, 21)
    g = F.GPUSolver2(m, p)
    g.set_state(U)
    it, _, _ = g.steady_solve(77, 0.0)
    assert it == 77 and g.resident_steps() == 75   # iterations 0 and 50 form the residual
    assert np.isfinite(g.get_state()).all()
    g.close()
