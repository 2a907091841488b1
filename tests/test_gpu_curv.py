"""Curvilinear FP64 kernel (csrc/curv.h) against the oracle: RHS and advance within 1e-12
(max-normalised per component, the bar of the FP64 form), at sizes around the 15 x 16 tile (one
tile and less, one row or column more, the smallest block, partial last tiles), with
wall-modelled faces on every axis; every chunk length gives the same cells."""
import numpy as np
import pytest

import cases
import golden_io
import oracle
from test_gpu_box import PARAMS, box_spec, state

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("needs a HIP device", allow_module_level=True)

import wmles_jax_amd as wmx  # noqa: E402


@pytest.mark.parametrize("n,walls,scheme,sgs", PARAMS)
def test_curvilinear_fp64_matches_the_oracle(n, walls, scheme, sgs):
    spec, arrays = box_spec(n, walls, scheme, sgs)
    X = arrays["nodes_all"]
    s = [2 * np.pi * X[d] / cases.L[d] for d in range(3)]
    arrays["nodes_all"] = X + 0.02 * min(cases.L) * np.stack(
        [np.sin(s[1]) * np.cos(s[2]), np.sin(s[0]) * np.cos(s[2]), np.cos(s[0]) * np.sin(s[1])])
    print(f"[curv fp64] {n}", flush=True)
    mesh, sol = cases.build(wmx, spec, arrays)
    _, ref = cases.build(oracle, spec, arrays)
    Q = state(mesh, sol)
    blk, ng = mesh.blocks[0], 3
    R = sol.rhs(Q)[0].cpu().numpy()
    assert golden_io.rel_err(blk.interior(R), blk.interior(ref.rhs(Q)[0])) <= 1e-12
    assert np.all(R[:, :ng] == 0.0) and np.all(R[:, :, :, -ng:] == 0.0)
    dt = float(sol.max_dt(Q))
    assert abs(dt - float(ref.max_dt(Q))) <= 1e-13 * dt
    assert golden_io.rel_err(sol.advance(Q, dt)[0].cpu().numpy(), ref.advance(Q, dt)[0]) <= 1e-12
    for ci in (1, 2, n[0]):
        sol.set_tiling(ci, 1)
        assert torch.equal(sol.rhs(Q)[0], torch.as_tensor(R, device="cuda"))
