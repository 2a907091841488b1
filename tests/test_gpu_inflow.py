"""Synthetic inflow rows around the forms of their row means (fewer than 9, 9..129 and more
spanwise cells), of the phase table (modes that do and do not divide the workgroup, rows too
large for it) and of the table search, against the oracle at the golden ramp's 1e-13."""
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


@pytest.mark.parametrize("nz,n_modes", [(4, 8), (8, 7), (9, 64), (33, 64), (129, 12), (131, 64), (300, 5)])
def test_inflow_rows_match_the_oracle(nz, n_modes):
    spec, arrays, prim = cases.ramp_spec(wmx, 12, 6, nz, n_modes=n_modes)
    ng = spec["ng"]
    _, s0 = cases.build(oracle, spec, arrays)
    _, s1 = cases.build(wmx, spec, arrays)
    Q = s1.init_state(prim)
    t = 0.05 * spec["ramp_props"]["L"] / spec["ramp_props"]["U_inf"]
    A = s1.apply_bcs(Q, s1.geoms, t)[0].cpu().numpy()
    B = np.asarray(s0.apply_bcs([q.cpu().numpy() for q in Q], s0.geoms, t)[0])
    assert golden_io.rel_err(A[:, :ng], B[:, :ng]) <= 1e-13


@pytest.mark.parametrize("nz,n_modes", [(694, 8), (1017, 5), (536, 11)])
def test_wide_rows_with_a_large_phase_table_match_the_oracle(nz, n_modes):
    """Rows of more than 512 cells whose phase table leaves room for one row buffer."""
    test_inflow_rows_match_the_oracle(nz, n_modes)
