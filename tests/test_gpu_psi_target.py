"""psi reads into every kind of memory: device buffers a kernel can write,
device addresses of 8 byte alignment, a range at the end of an allocation, host
memory, and between steps in flight."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [32, 512, 2048])
@pytest.mark.parametrize("dealiased", [False, True])
def test_psi_targets(N, dealiased):
    import torch
    from quantumvortices_amd import _native as nat, gpe as G
    rng = np.random.default_rng(N)
    psi = 1.0 + 0.1 * (rng.standard_normal((N, N)) + 1j * rng.standard_normal((N, N)))
    g = G.GPE(G.params_from_namelist(N, 1e-4, 2.5))
    g.set_psi(psi, sync=dealiased)
    if dealiased:
        g.rk4_async(2)      # the read waits for the steps
    host = np.empty((N, N), complex)
    nat.check(nat.lib().vk_gpe_get_psi(g.h, nat.ptr(host), None))
    if not dealiased:       # one transform there and back
        assert np.abs(host - psi).max() < 1e-13
    n = 2 * N * N
    for off in (0, 1, 2):   # in doubles; the buffer ends where the range does
        buf = torch.full((n + off,), 7.0, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        p = ctypes.cast(buf.data_ptr() + 8 * off, ctypes.POINTER(ctypes.c_double))
        nat.check(nat.lib().vk_gpe_get_psi(g.h, p, None))
        got = buf.cpu().numpy()
        assert np.all(got[:off] == 7.0)
        assert np.array_equal(got[off:].view(complex).reshape(N, N), host)
    # the staging of reads and writes and the steps' own rows share memory:
    # a write and a read between steps leave the field alone
    g.rk4_async(1)
    g.psi_to(host)
    k = g.kpsi
    g.rk4_async(1)
    h = G.GPE(G.params_from_namelist(N, 1e-4, 2.5))
    nat.check(nat.lib().vk_gpe_set_kpsi(h.h, nat.ptr(k)))
    h.gpe_rk4(1)
    assert np.array_equal(h.kpsi, g.kpsi)
    g.close()
    h.close()
