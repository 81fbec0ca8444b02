"""The gradient read into device memory is complete when the call returns,
whatever else the device's default stream is doing, and is the step's that came
before it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_device_gradient_is_of_the_step_before():
    import torch
    from quantumvortices_amd import _native as nat, warmstart as W
    print("case fno gradient order", flush=True)
    N = 128
    f = W.FNO(N, width=16, modes=8, layers=2, proj=16, cin=3, batch=2)
    f.set_params(f.init_params(3))
    rng = np.random.default_rng(7)

    def data():
        return (rng.standard_normal((2, 3, N, N)).astype(np.float32),
                rng.standard_normal((2, 2, N, N)).astype(np.float32))

    f.train_step(*data(), 0.0)
    first = f.grad()
    a = torch.zeros(f.nparams, dtype=torch.float32, device="cuda")
    b = torch.zeros_like(a)
    m = torch.full((4096, 4096), 1.0 / 4096, dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    for _ in range(40):     # tens of milliseconds on the default stream
        m = m @ m
    nat.check(nat.lib().vk_fno_get_grad(f.h, nat.fptr(a)))
    f.train_step(*data(), 0.0)
    nat.check(nat.lib().vk_fno_get_grad(f.h, nat.fptr(b)))
    torch.cuda.synchronize()
    assert np.array_equal(a.cpu().numpy(), first)
    assert np.array_equal(b.cpu().numpy(), f.grad())
    assert not np.array_equal(f.grad(), first)
    f.close()
