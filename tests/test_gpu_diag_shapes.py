"""The diagnostics at every pass shape, against the oracle: both states of a
field (dealiased, and with modes beyond the cutoff), without particles and with
them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def G():
    from quantumvortices_amd import gpe
    return gpe


@pytest.mark.parametrize("N", [32, 64, 256, 512, 1024, 2048])
@pytest.mark.parametrize("sync,npart", [(True, 0), (False, 0), (True, 3)])
def test_diagnostics_shapes(G, oracle_mod, N, sync, npart):
    O = oracle_mod
    rng = np.random.default_rng(N + npart)
    # no symmetry, waves up to beyond the cutoff
    k = np.zeros((N, N), complex)
    n = 12
    k[:n, :n] = 0.02 * (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n)))
    k[0, 0] = 1.0
    i = N // 2 - 3
    k[i, 2] = k[3, i] = k[i, i] = 0.01 + 0.02j
    psi = np.fft.ifft2(k) * N * N
    kw, okw = {}, {}
    if npart:
        kw = dict(gp_N_obj=npart, ppotV0=10.0, ppotd=1.5, gp_mass_part=5.0)
        okw = dict(np_=npart, V0_in=10.0, d_in=1.5, mass=5.0)
    g = G.GPE(G.params_from_namelist(N, 1e-3, 2.5, **kw))
    g.set_psi(psi, sync=sync)
    st = O.State(O.make_params(N, 1e-3, 2.5, **okw))
    st.set_psi(psi, sync=sync)
    if npart:
        pos = rng.uniform(0, 2 * np.pi, (npart, 2))
        vel = rng.uniform(-0.1, 0.1, (npart, 2))
        g.initialize_particles(pos, vel)
        st.part(0)[...] = pos
        st.part(1)[...] = vel
        st.particle_potential()
    d = g.diagnostics_gpe()
    scal, spec, pscal = st.diagnostics()
    print("N", N, "scal", d["scal"], scal, flush=True)
    # sums of one sign: relative; the momenta against the energies
    for i in (0, 1, 2, 3, 4):
        assert abs(d["scal"][i] - scal[i]) <= 1e-11 * abs(scal[i])
    for i in (5, 6):
        assert abs(d["scal"][i] - scal[i]) <= 1e-12 * (abs(scal[0]) + abs(scal[1]))
    for i in range(6):
        a, b = d["spec"][i], spec[i]
        assert np.linalg.norm(a - b) <= 1e-11 * np.linalg.norm(b)
    if npart:
        assert abs(d["eppot"] - pscal[0]) <= 1e-11 * abs(pscal[0])
    # the field is left as it was
    e = g.diagnostics_gpe()
    assert np.array_equal(e["scal"], d["scal"]) and np.array_equal(e["spec"], d["spec"])
    g.close()
