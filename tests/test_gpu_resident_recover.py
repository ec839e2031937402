"""Runs that the resident kernel cannot finish go on with the launched kernels from the state they had: a wait
between its work-groups that gives up (forced by a limit of 0 polls, with which every work-group leaves at its
first wait)."""
import numpy as np
import pytest

import cfd_solver_2d_gpu_amd as F
from helpers import vortex_case, wedge_case
from test_gpu_resident import naca_case

pytestmark = pytest.mark.gpu


def announce(msg):
    print(f"[gpu-case] {msg}", flush=True)


CASES = {
    "vortex_rk3": lambda: vortex_case(31),
    "wedge_euler": lambda: wedge_case(65, 33, scheme=F.SOL_ROE, advance=F.EVO_EXPLICIT),
    "wedge_mixed": lambda: wedge_case(65, 33, scheme=F.SOL_ROE, precision=F.PREC_MIXED),
}


def runs(m, p, U, polls):
    """State, time and step info of runs of 5, 6 and 7 steps; the second one with the given polls (None:
    launched kernels throughout)."""
    g = F.GPUSolver2(m, p)
    g.set_state(U)
    out, t = [], 0.0
    for k, n in enumerate((5, 6, 7)):
        if polls is None:
            g.use_resident(False)
        elif k == 1:
            g.use_resident(True, polls)
        t, info = g.advance(n, t, 1e9, F.NORM_INF)
        out += [g.get_state(), t, info.dt, info.t, info.n_restricted, np.array(info.residual[:]), g.stage_rhs()]
    steps = g.resident_steps()
    g.close()
    return out, steps


@pytest.mark.parametrize("case", list(CASES))
def test_run_goes_on_after_a_wait_that_gives_up(case):
    announce(f"a run whose waits give up at once: {case}")
    m, p, U = CASES[case]()
    want, n = runs(m, p, U, None)
    assert n == 0
    got, n = runs(m, p, U, 0)
    assert n == 5    # the run before; the handle stays with the launched kernels
    for a, b in zip(got, want):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("advance", [F.EVO_EXPLICIT, F.EVO_RK3])
def test_steady_solve_goes_on_after_a_wait_that_gives_up(advance):
    announce(f"pseudo-time iterations whose waits give up at once, time advance {advance}")
    m, p, U = naca_case(48, 21, time_advance=advance)
    out = []
    for polls in (None, 0):
        g = F.GPUSolver2(m, p)
        g.set_state(U)
        res = []
        for k, n in enumerate((60, 77, 130)):
            if polls is None:
                g.use_resident(False)
            elif k == 1:
                g.use_resident(True, polls)
            it, r0, r = g.steady_solve(n, 0.0)
            res += [it, r0, r, g.get_state()]
        assert g.resident_steps() == (0 if polls is None else 58)
        # and the handle serves other calls as before
        t, info = g.advance(5, 0.0, 1e9, F.NORM_2)
        res += [t, info.dt, np.array(info.residual[:]), g.get_state()]
        if polls is not None:
            g.use_resident(True)
            g.set_state(res[3])
            g.steady_solve(77, 0.0)
            assert g.resident_steps() == 58 + 75
            assert np.array_equal(g.get_state(), res[7])
        g.close()
        out.append(res)
    for a, b in zip(*out):
        assert np.array_equal(a, b)


def test_batch_of_one_case_goes_on_after_a_wait_that_gives_up():
    announce("a batch of one case whose waits give up at once")
    m, p, U = wedge_case(65, 33, scheme=F.SOL_ROE)
    out = []
    for polls in (-1, 0):
        b = F.BatchSolver([m], [p])
        F.check(F.lib().fvmr_use_resident(b._h, 1, polls), "fvmr_use_resident")
        b.set_state(0, U)
        t = b.advance(6, np.zeros(1), np.full(1, 1e9))
        t = b.advance(6, t, np.full(1, 1e9))
        out.append((b.get_state(0), t))
        b.close()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
