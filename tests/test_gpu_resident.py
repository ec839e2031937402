"""The resident kernel (many steps of a small mesh in one launch) against the launched kernels: a run of
n steps equals n single steps, which the launched kernels do, bit for bit: fields, time, time step and
residual norms; so do pseudo-time iterations.  Tile sizes put the number of work-groups at one, at a few, near
what fits on the device and beyond it."""
import threading

import numpy as np
import pytest

import cfd_solver_2d_gpu_amd as F
from helpers import cylinder_case, vortex_case, wedge_case

pytestmark = pytest.mark.gpu


def announce(msg):
    print(f"[gpu-case] {msg}", flush=True)


def triangle_case():
    """One triangle with three farfield faces: one tile, no halo."""
    m = F.Mesh.from_lists([0.0, 1.0, 0.2], [0.0, 0.1, 0.9], [0, 1, 2], [5], [[0, 1, 2]], [("far", [(0, 1), (1, 2), (2, 0)])])
    p = F.default_params(inf_ruvp=[1.0, 0.4, 0.1, 1.0], CFL=0.5)
    U = F.field_init(m, p)
    U[0] *= 1.1
    return m, p, U


def naca_case(ni, nj, **kw):
    m = F.Mesh.generate(F.GEN_NACA_OGRID, ni, nj, b=20.0, c=1.05, naca_digits=12)
    inf = list(F.ruvp_from_mach(0.5, 2.0))
    p = F.default_params(inf_ruvp=inf, inlet_ruvp=inf, outlet_ruvp=inf, CFL=1.0, venkat_K=5.0,
                         limiter=F.LIM_VENKATAKRISHNAN, **kw)
    return m, p, F.field_init(m, p)


def both(m, p, U, n, T=1e9, norm=F.NORM_INF):
    """(state, t, dt, residual, restricted) after one advance of n steps and after n single steps."""
    out = []
    for whole in (True, False):
        g = F.GPUSolver2(m, p)
        g.set_state(U)
        t = 0.0
        if whole:
            t, info = g.advance(n, t, T, norm)
        else:
            for _ in range(n):
                t, info = g.iteration_device(t, T, norm)
        out.append((g.get_state(), t, info.dt, np.array(info.residual[:]), info.n_restricted))
        g.close()
    return out


def same(a, b):
    assert a[1] == b[1] and a[2] == b[2] and a[4] == b[4]
    assert np.array_equal(a[3], b[3], equal_nan=True)
    assert np.array_equal(a[0], b[0], equal_nan=True)


CASES = {
    "triangle": lambda gd: triangle_case(),
    "vortex_rk3_periodic": lambda gd: vortex_case(23),
    "vortex_euler_lsq_llf": lambda gd: vortex_case(31, gradient=F.GRA_LEASTSQUARE, scheme=F.SOL_LLF,
                                                   limiter=F.LIM_VENKATAKRISHNAN, advance=F.EVO_EXPLICIT),
    "wedge_roe_rk3": lambda gd: wedge_case(65, 33, scheme=F.SOL_ROE),
    "cylinder_viscous_euler": lambda gd: cylinder_case(gd),
}


@pytest.mark.parametrize("precision", [F.PREC_FP64, F.PREC_MIXED])
@pytest.mark.parametrize("case", list(CASES))
def test_run_equals_single_steps(case, precision, golden_dir):
    announce(f"resident run against single steps: {case}, precision {precision}")
    m, p, U = CASES[case](golden_dir)
    p.precision = precision
    for n in (4, 9):
        same(*both(m, p, U, n))


@pytest.mark.parametrize("tile_cells", [1, 2, 3, 61])
def test_run_equals_single_steps_over_tile_counts(tile_cells):
    announce(f"resident run against single steps: tiles of {tile_cells} cells")
    m, p, U = wedge_case(45, 22, scheme=F.SOL_ROE)   # 1,980 cells: 1,980, 990, 660 and 33 tiles
    p.tile_cells = tile_cells
    same(*both(m, p, U, 7))


def test_run_stops_at_the_end_time():
    announce("resident run across its end time")
    m, p, U = wedge_case(40, 20, scheme=F.SOL_ROE)
    g = F.GPUSolver2(m, p)
    g.set_state(U)
    t, _ = g.advance(5, 0.0, 1e9)
    g.close()
    a, b = both(m, p, U, 12, T=0.9 * t)   # dt is clamped in step 5 and 0 after it
    same(a, b)
    assert a[1] == 0.9 * t and a[2] == 0.0


@pytest.mark.parametrize("n", [6, 20])
def test_run_with_cells_to_restrict(n):
    announce(f"resident run with cells to restrict, {n} steps")
    m, p, U = wedge_case(40, 20, scheme=F.SOL_ROE)
    U[0, 700] = 400.0       # out of range: restricted after the first step
    U[3, 1201] = np.nan
    same(*both(m, p, U, n))


@pytest.mark.parametrize("advance", [F.EVO_EXPLICIT, F.EVO_RK3])
def test_steady_iterations_equal_single_ones(advance):
    announce(f"resident pseudo-time iterations against single ones, time advance {advance}")
    m, p, U = naca_case(48, 21, time_advance=advance)
    out = []
    for whole in (True, False):
        g = F.GPUSolver2(m, p)
        g.set_state(U)
        if whole:
            it, _, _ = g.steady_solve(77, 0.0)
            assert it == 77
        else:
            for _ in range(77):
                g.steady_solve(1, 0.0)
        out.append(g.get_state())
        g.close()
    assert np.array_equal(*out)


def test_two_threads():
    announce("resident runs of two handles from two threads")
    cases = [wedge_case(100, 50, scheme=F.SOL_ROE), vortex_case(60)]
    want = [both(m, p, U, 50)[0] for m, p, U in cases]
    got, errors = [None, None], []

    def work(k):
        try:
            m, p, U = cases[k]
            g = F.GPUSolver2(m, p)
            for _ in range(10):
                g.set_state(U)
                t, info = g.advance(50, 0.0, 1e9, F.NORM_INF)
            got[k] = (g.get_state(), t, info.dt, np.array(info.residual[:]), info.n_restricted)
            g.close()
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
    for a, b in zip(got, want):
        same(a, b)
