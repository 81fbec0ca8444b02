"""The network's row kernels at the edges of their tiles: one to nine chunks
of 64 columns per row (fewer chunks than waves, a remainder over the waves,
two rounds), every (width, modes), one layer (the lift feeds the projection
directly) and several, hidden widths off the 16-row tiles, one to four input
planes, batches smaller than the handle's.  Output, loss and gradient against
the float64 oracle on the same BF16 weights.

Tolerances, from the arithmetic: products and sums are FP32 (2^-24 = 6e-8 per
rounding); a value passes about four contractions per layer whose blocked
sums chain at most ~200 roundings (16 matrix steps of 4, then chunks, waves,
workgroups), a random walk of sqrt(200) 6e-8 = 8e-7 each, so 2e-5 for the
output of four layers, and twice that again for a gradient."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

CASES = [  # N, width, modes, layers, proj, cin, nb, batch
    (64, 32, 16, 1, 64, 3, 1, 1),
    (64, 8, 4, 2, 7, 1, 3, 4),
    (192, 16, 8, 2, 17, 4, 2, 2),
    (192, 32, 16, 2, 1, 2, 1, 3),
    (320, 8, 4, 3, 64, 3, 1, 1),
    (320, 32, 16, 1, 33, 3, 2, 2),
    (576, 16, 8, 1, 16, 3, 1, 1),
]


@pytest.mark.parametrize("N,width,modes,layers,proj,cin,nb,batch", CASES)
def test_row_kernels_match_oracle(N, width, modes, layers, proj, cin, nb, batch):
    import torch
    assert torch.cuda.is_available()
    import fno_oracle as FO
    from quantumvortices_amd import warmstart as W
    print("case fno rows", N, width, modes, layers, proj, cin, nb, batch, flush=True)
    f = W.FNO(N, width=width, modes=modes, layers=layers, proj=proj, cin=cin, batch=batch)
    p = f.init_params(N + layers)
    for l in range(layers):
        o, n = f.blocks["R%d" % l]
        p[o:o + n] *= 2.0 * width      # the spectral path carries signal
    rng = np.random.default_rng(N + proj)
    for b in ["bp", "bq1", "bq2"] + ["b%d" % l for l in range(layers)]:
        o, n = f.blocks[b]
        p[o:o + n] = rng.normal(0.0, 0.1, n)
    f.set_params(p)
    p = f.get_params().astype(np.float64)
    x = rng.standard_normal((nb, cin, N, N)).astype(np.float32)
    t = rng.standard_normal((nb, 2, N, N)).astype(np.float32)
    ref, _ = FO.forward(p, x.astype(np.float64), f.dims)
    assert rel_l2(f.forward(x), ref) < 2e-5
    loss = f.train_step(x, t, lr=0.0)
    lref, gref = FO.loss_grad(p, x.astype(np.float64), t.astype(np.float64), f.dims)
    assert abs(loss - lref) < 4e-5 * lref
    assert rel_l2(f.grad(), gref) < 4e-5
    assert rel_l2(f.forward(x), ref) < 2e-5     # after a training step, the same
    f.close()


def test_gelu_limits():
    """Zero weights leave the bias of the projection's hidden units, so the
    output is Q2 gelu(bq1): the activation over its whole range, to an FP32
    ulp of the larger of |x Phi(x)| and |x| 2^-24 (Phi's absolute error)."""
    import math
    from quantumvortices_amd import warmstart as W
    xs = np.concatenate([np.linspace(-12.0, 12.0, 97), [0.0, 1e-6, -1e-6, 30.0, -30.0, 100.0, -100.0]])
    f = W.FNO(64, width=8, modes=4, layers=1, proj=1, cin=1, batch=1)
    for v in xs:
        p = np.zeros(f.nparams, dtype=np.float32)
        p[f.blocks["bq1"][0]] = v
        p[f.blocks["Q2"][0]] = 1.0
        f.set_params(p)
        u = float(f.get_params()[f.blocks["bq1"][0]])      # BF16
        y = f.forward(np.zeros((1, 1, 64, 64), dtype=np.float32))
        ref = 0.5 * u * math.erfc(-u / math.sqrt(2.0))
        assert abs(float(y[0, 0, 5, 7]) - ref) <= 2.0 ** -23 * abs(ref) + 2.0 ** -24 * abs(u), u
        assert np.all(y[0, 0] == y[0, 0, 0, 0]) and np.all(y[0, 1] == 0.0)
    f.close()
