"""Graphs and the resident kernel: with both allowed a run is resident; replays of the launched kernels (resident
kernel off) give the fields of eager launches, replay after replay, with eager work and host
synchronisations in between."""
import numpy as np
import pytest

import cfd_solver_2d_gpu_amd as F
from helpers import vortex_case, wedge_case

pytestmark = pytest.mark.gpu


def announce(msg):
    print(f"[gpu-case] {msg}", flush=True)


CASES = {
    "vortex_fp64": lambda: vortex_case(48),
    "wedge_mixed": lambda: wedge_case(64, 32, scheme=F.SOL_ROE, precision=F.PREC_MIXED),
}


@pytest.mark.parametrize("case", list(CASES))
def test_graphs_leave_the_resident_kernel_on(case):
    announce(f"resident runs of a handle with graphs: {case}")
    m, p, U = CASES[case]()
    out = []
    for on in (False, True):
        g = F.GPUSolver2(m, p)
        g.use_graphs(on)
        g.set_state(U)
        t = 0.0
        for n in (7, 3, 12):
            t, _ = g.advance(n, t, 1e9)
        assert g.resident_steps() == 19
        out.append((t, g.get_state()))
        g.close()
    assert out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("case", list(CASES))
def test_graph_replays_of_the_launched_kernels(case):
    announce(f"graph replays vs eager launches: {case}")
    m, p, U = CASES[case]()
    gs, ts = [], [0.0, 0.0]
    for on in (False, True):
        g = F.GPUSolver2(m, p)
        g.use_resident(False)
        g.use_graphs(on)
        g.set_state(U)
        gs.append(g)
    for n, norm in ((7, 0), (3, F.NORM_INF), (6, 0), (4, F.NORM_2), (13, F.NORM_1)):
        infos = []
        for k, g in enumerate(gs):
            ts[k], info = g.advance(n, ts[k], 1e9, residual_norm=norm)
            infos.append(np.array(info.residual[:]) if norm else 0)
        assert ts[0] == ts[1] and np.array_equal(*infos)
        assert np.array_equal(gs[0].get_state(), gs[1].get_state())
        for g in gs:
            g.stage_rhs()
    for g in gs:
        assert g.resident_steps() == 0
        g.close()
