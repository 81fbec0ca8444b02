"""The particles' update as the first workgroups of P4's launch (up to 1024^2)
against the update in a launch of its own, which timed passes keep: the same
bits, for particle counts around the multiples of eight it is padded to."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,npart", [(32, 3), (64, 1), (128, 7), (128, 8), (256, 9), (512, 16), (512, 17), (1024, 5),
                                     (2048, 3)])
def test_update_with_p4_equals_update_alone(N, npart):
    from quantumvortices_amd import gpe as G
    rng = np.random.default_rng(N + npart)
    x = np.arange(N) * 2.0 * np.pi / N
    psi = 1.0 + 0.1 * np.exp(1j * (x[None, :] + 2 * x[:, None])) + 0.05 * np.cos(3 * x)[None, :]
    pos, vel = rng.uniform(0.0, 2.0 * np.pi, (npart, 2)), rng.normal(0.0, 0.1, (npart, 2))
    out = []
    for timed in (False, True):
        g = G.GPE(G.params_from_namelist(N, 1e-3, 2.5, gp_N_obj=npart, ppotV0=10.0, ppotd=2.0, gp_mass_part=0.5))
        g.set_psi(psi, sync=True)
        g.initialize_particles(pos, vel)
        if timed:
            g.pass_times(3)
        else:
            g.gpe_rk4(3)
        out.append((g.kpsi, *g.particles()))
        g.close()
    print("N", N, "np", npart, "moved", np.abs(out[0][2] - vel).max(), flush=True)
    assert np.abs(out[0][2] - vel).max() > 0.0
    for a, b in zip(*out):
        assert np.array_equal(a, b)
