"""Runs that the resident kernel cannot finish go on with the launched kernels from the state they had: a wait
between its work-groups that gives up (forced by a limit of 0 polls, with which every work-group leaves at its
first wait) and a cooperative launch or an allocation that the device refuses (a child process with a layer in front of
the runtime's calls)."""
import os
import subprocess
import sys

import numpy as np
import pytest

import cfd_solver_2d_gpu_amd as F
from cfd_solver_2d_gpu_amd.build import C_API_DIR
from conftest import ROOT
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


REFUSED = r"""
import ctypes as C, sys
sys.path[:0] = [sys.argv[2], sys.argv[2] + "/tests"]
front = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)   # before the library, which then calls it
import numpy as np
import cfd_solver_2d_gpu_amd as F
from helpers import wedge_case
from test_gpu_resident import naca_case

def var(name):
    return C.c_int.in_dll(front, name)

def run(case, launched=False):
    m, p, U = case()
    g = F.GPUSolver2(m, p)
    g.use_resident(not launched)
    g.set_state(U)
    out = []
    t = 0.0
    for _ in range(2):
        t, info = g.advance(9, t, 1e9, F.NORM_INF)
        out += [g.get_state(), t, info.dt, np.array(info.residual[:])]
    if p.limiter == F.LIM_VENKATAKRISHNAN:
        out += [*g.steady_solve(77, 0.0), g.get_state()]
    n = g.resident_steps()
    g.close()
    return out, n

cases = {"wedge": lambda: wedge_case(65, 33, scheme=F.SOL_ROE), "naca": lambda: naca_case(48, 21)}
for name, case in cases.items():
    want, n = run(case, launched=True)
    assert n == 0
    got, n = run(case)   # resident, unless the device itself refuses: this process is its second one here
    assert var("refused").value == 0
    assert all(np.array_equal(a, b) for a, b in zip(got, want))
    if sys.argv[3] == "launch":
        var("refuse_cooperative").value = 1
    else:   # the last allocation of a handle's creation: the resident kernel's
        m, p, U = case()
        var("mallocs").value = 0
        F.GPUSolver2(m, p).close()
        var("refuse_malloc").value = var("mallocs").value
        var("mallocs").value = 0
    got, n = run(case)
    assert n == 0 and var("refused").value >= 1
    assert all(np.array_equal(a, b) for a, b in zip(got, want))
    for v in ("refuse_cooperative", "refuse_malloc", "refused"):
        var(v).value = 0
    print("ok", name, flush=True)
"""


@pytest.fixture(scope="module")
def front(tmp_path_factory):
    """The layer in front of the runtime (tests/c_api/hip_refuse.cpp)."""
    out = str(tmp_path_factory.mktemp("front") / "libhip_refuse.so")
    rocm = "/opt/rocm"
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", f"-I{rocm}/include",
                    os.path.join(C_API_DIR, "hip_refuse.cpp"), f"-L{rocm}/lib", "-Wl,--no-as-needed", "-lamdhip64",
                    f"-Wl,-rpath,{rocm}/lib", "-o", out], check=True)
    return out


def refused(front, what):
    r = subprocess.run([sys.executable, "-c", REFUSED, front, ROOT, what], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.split() == ["ok", "wedge", "ok", "naca"], r.stdout + r.stderr


def test_refused_launch_goes_on_with_the_launched_kernels(front):
    announce("cooperative launches that the device refuses")
    refused(front, "launch")


def test_refused_allocation_leaves_the_launched_kernels(front):
    announce("the resident kernel's memory refused at creation")
    refused(front, "memory")
