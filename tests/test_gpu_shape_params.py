"""Parameters changed on a handle in its second transform shape (an ensemble of
one, whose member table holds them on the device): the steps that follow are those
of a fresh handle with these parameters, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _field(N):
    rng = np.random.default_rng(N)
    return 1.0 + 0.1 * (rng.standard_normal((N, N)) + 1j * rng.standard_normal((N, N)))


@pytest.mark.parametrize("N", [256, 512, 1024])
def test_set_dt_in_shape_1(N):
    from quantumvortices_amd import gpe as G
    a = G.GPE(G.params_from_namelist(N, 2e-4, 2.5))
    a.set_shape(1)
    a.set_psi(_field(N), sync=True)
    a.gpe_rk4(2)
    k = a.kpsi
    a.set_dt(1e-4)
    a.gpe_rk4(2)
    b = G.GPE(G.params_from_namelist(N, 1e-4, 2.5))
    b.set_shape(1)
    b.set_kpsi(k)
    b.gpe_rk4(2)
    assert np.array_equal(a.kpsi, b.kpsi)
    a.close()
    b.close()


@pytest.mark.parametrize("N", [256, 1024])
def test_chemical_potential_in_shape_1(N):
    """RK4 after SGLE runs at the chemical potential that SGLE reached."""
    from quantumvortices_amd import gpe as G
    a = G.GPE(G.params_from_namelist(N, 2e-4, 2.5))
    a.set_shape(1)
    a.set_psi(_field(N), sync=True)
    a.gpe_rk4(1)
    a.set_sgle(True, oneybeta=1e-7, nuN=0.5, seed=3)
    a.ARGLE(nsteps=3)
    om = a.chempot
    k = a.kpsi
    a.gpe_rk4(2)
    p = G.params_from_namelist(N, 2e-4, 2.5)
    assert om != p.omega
    p.omega = om
    b = G.GPE(p)
    b.set_shape(1)
    b.set_kpsi(k)
    b.gpe_rk4(2)
    assert np.array_equal(a.kpsi, b.kpsi)
    a.close()
    b.close()
