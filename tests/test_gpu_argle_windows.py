"""ARGLE around obstacles at sizes on both sides of the line between the
potential on the grid and the window tables in P3, plain and advective, obstacles
at the edges of the box and on top of each other: kpsi and the residual against the
oracle's spectral translation, to the bound of the other ARGLE comparisons (the
potential's spectrum beyond the dealias radius, 1e-24 of its peak, is far below)."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,tg", [(1024, 0), (1024, 1), (2048, 0), (2048, 1), (4096, 0)])
def test_argle_obstacles_vs_oracle(oracle_mod, N, tg):
    from quantumvortices_amd import gpe as G
    print("case argle windows", N, tg, flush=True)
    O = oracle_mod
    dt, n = 1e-2, 4
    dx = 2 * np.pi / N
    x = np.arange(N) * dx
    psi = 1.0 + 0.1 * np.exp(1j * (x[None, :] + 2 * x[:, None])) + 0.05 * np.cos(3 * x)[None, :]
    pos = np.array([[0.0, 0.0], [5 * dx, (N - 1) * dx], [-0.7, 2 * np.pi + 0.4], [5 * dx, (N - 1) * dx + 3 * dx]])
    p = G.params_from_namelist(N, dt, 2.5, gp_N_obj=n, ppotV0=10.0, ppotd=2.0, gp_mass_part=1.0)
    g = G.GPE(p)
    if tg:
        g.set_advection(True, 0.3, -0.2)
    g.set_psi(psi, sync=False)
    g.set_obstacles(pos, 10.0 * p.g, 2.0 * p.xi)
    kw = dict(adv=1, vnx=0.3, vny=-0.2) if tg else {}
    st = O.State(O.make_params(N, dt, 2.5, np_=n, V0_in=10.0, d_in=2.0, mass=1.0, **kw))
    st.set_psi(psi, sync=False)
    st.part(0)[...] = pos
    st.particle_potential()
    r, ro = g.ARGLE(nsteps=2), st.argle(2)
    assert rel_l2(g.kpsi, st.kpsi) < 1e-11 and abs(r - ro) <= 1e-9 * abs(ro)
    # another set of obstacles, the same handle
    g.set_psi(psi, sync=False)
    g.set_obstacles(pos[:2] + 0.3, 10.0 * p.g, 2.0 * p.xi)
    h = G.GPE(p)
    if tg:
        h.set_advection(True, 0.3, -0.2)
    h.set_psi(psi, sync=False)
    h.set_obstacles(pos[:2] + 0.3, 10.0 * p.g, 2.0 * p.xi)
    assert g.ARGLE(nsteps=2) == h.ARGLE(nsteps=2)
    assert np.array_equal(g.kpsi, h.kpsi)
    g.close()
    h.close()
