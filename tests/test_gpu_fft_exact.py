"""The small bins beside a large one: differences of nearly equal halves of a
transform are exact.  Input that alternates between 1 and 1 + 2^-52 along an axis
(or both) has two bins per axis; the Nyquist one is a multiple of 2^-52 that a
double holds, formed by sums of equal values (exact) and one difference of
neighbours (exact), while the sum of the same neighbours does not fit a double.
Every other bin is a sum of zeros.  So the transform has to give the Nyquist bin
and the zeros exactly, whatever its size and shape; the inverse likewise."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

U = 2.0 ** -52


@pytest.mark.parametrize("N", [32, 64, 128, 256, 512, 1024, 2048, 4096])
@pytest.mark.parametrize("axis", ["x", "y", "xy"])
def test_nyquist_bin_beside_the_mean(N, axis):
    from quantumvortices_amd import _native as nat, gpe as G
    print("case exact bins", N, axis, flush=True)
    par = np.arange(N) % 2
    odd = {"x": par[None, :] + 0 * par[:, None], "y": par[:, None] + 0 * par[None, :],
           "xy": (par[None, :] + par[:, None]) % 2}[axis]
    x = (1.0 + U * odd).astype(complex)      # [y, x]
    at = {"x": (N // 2, 0), "y": (0, N // 2), "xy": (N // 2, N // 2)}[axis]     # [kx, ky]
    g = G.GPE(G.params_from_namelist(N, 1e-3, 2.5))
    out = np.empty((N, N), complex)
    for sign, scale in ((-1, 1.0), (1, 1.0 / (float(N) * N))):
        a = x if sign < 0 else np.ascontiguousarray(x.T)        # k-space is [kx, ky]
        nat.check(nat.lib().vk_fft2d(g.h, sign, nat.dptr(np.ascontiguousarray(a)), nat.dptr(out)))
        f = out if sign < 0 else out.T       # [kx, ky], and for the inverse [x, y]
        assert f[at] == -0.5 * U * N * N * scale
        assert abs(f[0, 0] - N * N * scale) <= 4 * U * N * N * scale
        rest = np.abs(f)
        rest[at] = rest[0, 0] = 0.0
        assert not rest.any()
    g.close()
