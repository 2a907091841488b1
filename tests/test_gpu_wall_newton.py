"""Spalding's Newton loop stops early where its update returns its input, or the value
before it: every count must still give what the full loop gives."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("needs a HIP device", allow_module_level=True)

import wmles_jax_amd as wmx  # noqa: E402


def newton(h, U, rho, mu, n_iter, k=0.41, B=5.2):
    Reh = h * U * rho / mu
    up = np.clip(np.sqrt(Reh), 1.0, 25.0)
    for _ in range(n_iter):
        ku = k * up
        p2 = np.exp(ku) - 1.0 - ku - 0.5 * ku * ku
        F = up + np.exp(-k * B) * (p2 - ku ** 3 / 6.0) - Reh / up
        dF = 1.0 + np.exp(-k * B) * k * p2 + Reh / up ** 2
        up = np.clip(up - F / dF, 0.5 * up, 100.0)
    return U / up


@pytest.mark.parametrize("n", [1, 64, 4097])
def test_every_iteration_count_gives_the_full_loop(n):
    rng = np.random.default_rng(n)
    h, U, rho, mu = 10.0 ** rng.uniform(-4, -1, n), 10.0 ** rng.uniform(0, 2, n), np.full(n, 1.2), np.full(n, 1.8e-5)
    counts = list(range(1, 15)) + [29, 30, 41]
    got = {c: wmx.EquilibriumWallModel(n_iter=c).utau(h, U, rho, mu).cpu().numpy() for c in counts}
    for c in counts:
        assert np.allclose(got[c], newton(h, U, rho, mu, c), rtol=1e-13, atol=0.0)
    # once a face is at a fixed value or in a pair, the later counts hold the same value or the
    # pair's member of their parity, bit for bit
    done = (got[11] == got[13]) & (got[12] == got[14])
    assert done.mean() > 0.99
    for c in (29, 30, 41):
        assert np.array_equal(got[c][done], got[13 if c % 2 else 14][done])
    if n > 1000:
        assert np.any(got[13][done] != got[14][done])           # (pairs do occur)
