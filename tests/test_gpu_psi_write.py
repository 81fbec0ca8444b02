"""A psi written between steps that are still queued: the x-space buffer that
stages it is the one those steps pass their rows through, so the write has to wait
its turn on the handle's stream.  The steps after it start from the new field."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [64, 512, 2048])
@pytest.mark.parametrize("where", ["host", "device"])
def test_write_between_queued_steps(N, where):
    import torch
    from quantumvortices_amd import gpe as G
    rng = np.random.default_rng(N)
    f = [1.0 + 0.1 * (rng.standard_normal((N, N)) + 1j * rng.standard_normal((N, N))) for _ in range(2)]
    src = [torch.from_numpy(x).cuda() for x in f] if where == "device" else f
    torch.cuda.synchronize()
    g = G.GPE(G.params_from_namelist(N, 1e-4, 2.5))
    h = G.GPE(G.params_from_namelist(N, 1e-4, 2.5))

    def put(x, i):
        (x.set_psi_from if where == "device" else x.set_psi)(src[i], sync=True)

    put(g, 0)
    g.rk4_async(20)
    put(g, 1)
    g.rk4_async(1)
    put(h, 1)
    h.gpe_rk4(1)
    assert np.array_equal(g.kpsi, h.kpsi)
    assert np.array_equal(g.psi, h.psi)
    g.close()
    h.close()
