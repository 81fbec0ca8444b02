"""RK4 steps with real-space particles recorded into a graph on the handle's
stream: particles set between replays are the ones that the next replay starts
from (positions, windows and factor tables alike), bit for bit as with steps
that are launched."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N, NP = 256, 3


def _handle():
    from quantumvortices_amd import gpe as G
    p = G.params_from_namelist(N, 1e-3, 2.5, gp_N_obj=NP, ppotV0=10.0, ppotd=2.0, gp_mass_part=0.05)
    g = G.GPE(p)
    xs, ys, qs = G.lattice_vortices(4)
    g.set_psi(G.ic_vortices_host(N, xs, ys, qs, p.xi), sync=True)
    return g


def _state(g):
    return [g.kpsi] + [np.asarray(a) for a in g.particles()]


def test_particles_set_between_replays():
    from quantumvortices_amd import _native as nat
    print("case recorded steps", flush=True)
    L = nat.lib()
    v = ctypes.c_void_p
    rng = np.random.default_rng(5)
    where = [(rng.uniform(0.0, 2 * np.pi, (NP, 2)), rng.normal(0.0, 0.05, (NP, 2)), np.zeros((NP, 2)))
             for _ in range(3)]
    g, e = _handle(), _handle()
    for h in (g, e):
        h.initialize_particles(*where[0])
        h.gpe_rk4(1)
    stream = v(L.vk_gpe_stream(g.h))
    graph, run = v(), v()
    assert L.hipStreamBeginCapture(stream, 1) == 0
    g.rk4_async(1)
    assert L.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
    assert L.hipGraphInstantiate(ctypes.byref(run), graph, v(), v(), ctypes.c_size_t(0)) == 0
    for w in [None] + where[1:]:
        if w is not None:
            g.initialize_particles(*w)
            e.initialize_particles(*w)
        for _ in range(2):
            assert L.hipGraphLaunch(run, stream) == 0
            assert L.hipStreamSynchronize(stream) == 0
            e.gpe_rk4(1)
            for a, b in zip(_state(g), _state(e)):
                assert np.array_equal(a, b)
    assert L.hipGraphExecDestroy(run) == 0 and L.hipGraphDestroy(graph) == 0
    g.close()
    e.close()
