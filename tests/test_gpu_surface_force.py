"""Surface forces of sets around the 64 edges that a wave forms at a time: bit for bit the oracle's sums."""
import numpy as np
import pytest

import cfd_solver_2d_gpu_amd as F
import oracle as O

pytestmark = pytest.mark.gpu


def test_set_sizes_around_a_wave():
    print("[gpu-case] surface force of sets of 0, 1, 63, 64, 65, 128 and 200 edges", flush=True)
    m = F.Mesh.generate(F.GEN_CYLINDER_OGRID, 256, 20, a=0.5, b=10.0, c=1.1)
    inf = list(F.ruvp_from_mach(0.4, 3.0))
    p = F.default_params(inf_ruvp=inf, inlet_ruvp=inf, outlet_ruvp=inf)
    U = F.field_init(m, p)
    xy = m.arrays()["element_xy"]
    U[3] *= 1.0 + 0.05 * np.sin(3 * xy[0]) * np.cos(2 * xy[1])
    edges = np.concatenate([np.asarray(e, dtype=np.int32) for _, _, e in m.boundary_sets()])
    sets = [edges[:0], edges[5:6], edges[7:70], edges[3:67], edges[1:66], edges[100:228][::-1], edges[11:211]]
    g = F.GPUSolver2(m, p)
    g.set_state(U)
    _, cp, _ = g.node_field()
    got = g.surface_force(0.7, sets)
    direct = g.surface_force_noalloc(0.7, sets)
    g.close()
    want = O.surface_force(m.soa, cp, sets, 0.7)
    for a, b, c in zip(got, direct, want):
        assert np.array_equal(a, c) and np.array_equal(b, c)
