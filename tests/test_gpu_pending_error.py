"""A pending error of the runtime (as a failed launch among queued steps leaves
one) is reported by the next psi read, into host and into device memory, and by
that one alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("where", ["host", "device"])
def test_psi_read_reports_pending_error(where):
    import torch
    from quantumvortices_amd import _native as nat, gpe as G
    print("case pending error", where, flush=True)
    N = 64
    g = G.GPE(G.params_from_namelist(N, 1e-3, 2.5))
    g.set_psi(np.ones((N, N), complex), sync=True)
    g.rk4_async(1)
    host = np.zeros((N, N), complex)
    dev = torch.zeros((N, N), dtype=torch.complex128, device="cuda")
    torch.cuda.synchronize()
    out = nat.ptr(host) if where == "host" else nat.dptr(dev)
    # the library's own runtime: a device number that does not exist is refused by the host
    assert nat.lib().hipSetDevice(1 << 20) != 0
    with pytest.raises(nat.VKError):
        nat.check(nat.lib().vk_gpe_get_psi(g.h, out, None))
    nat.check(nat.lib().vk_gpe_get_psi(g.h, out, None))
    got = host if where == "host" else dev.cpu().numpy()
    assert np.abs(np.abs(got) - 1.0).max() < 1e-12
    g.close()
