"""The mass-flux constraint on either side of the 64 partials (of 1024 cells) up to which its last
sum rides in the launch that applies it, against the oracle."""
import numpy as np
import pytest

import cases
import golden_io
import oracle

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("needs a HIP device", allow_module_level=True)

import wmles_jax_amd as wmx  # noqa: E402


@pytest.mark.parametrize("nblocks,n", [(1, (6, 4, 4)), (1, (64, 32, 32)), (1, (65, 32, 32)), (2, (40, 24, 24)), (3, (99, 32, 32))])
def test_mass_flux_matches_the_oracle(nblocks, n):
    splits = [round(b * n[0] / nblocks) for b in range(nblocks + 1)]
    spec, arrays = cases.channel_spec(nblocks, *n, {"kind": "KEP", "order": 2}, "none", splits=splits)
    m0, s0 = cases.build(oracle, spec, arrays)
    _, s1 = cases.build(wmx, spec, arrays)
    pr = spec["props"]
    Q = cases.interior_noise(m0.blocks, s0.init_state(lambda xc: cases.channel_prim(xc, pr, 3)), 4, 0.05)
    c0, c1 = s0.constraints[0], s1.constraints[0]
    A = [np.asarray(q.cpu()) for q in c1(tuple(torch.as_tensor(q, device="cuda") for q in Q), s1.geoms, s1.blocks)]
    for a, b in zip(A, c0(Q, s0.geoms, s0.blocks)):
        assert golden_io.rel_err(a, b) <= 1e-13
    dt = float(s0.max_dt(Q)) * 0.5
    for a, b, blk in zip(s1.advance(Q, dt), s0.advance(Q, dt), m0.blocks):
        assert golden_io.rel_err(a.cpu().numpy(), b) <= 1e-12
