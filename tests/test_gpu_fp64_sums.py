"""FP64 outward sums where the flow does not change along i: the two i faces of a cell carry the same
pressure-sized flux, and what is left of the x momentum is the viscous force, 1e-9 of it.  Summed
through the pressure it would keep eight digits; the bar is the form's 1e-12."""
import numpy as np
import pytest

import cases
import oracle
from test_gpu_box import box_spec

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("needs a HIP device", allow_module_level=True)

import wmles_jax_amd as wmx  # noqa: E402


def shear(xc):
    """rho 1, p 1e5, u(y, z) alone: every product with the density is exact."""
    u = 0.5 * np.sin(2 * np.pi * xc[1] / cases.L[1]) * np.cos(2 * np.pi * xc[2] / cases.L[2])
    one = np.ones_like(u)
    return np.stack([one, u, 0.0 * u, 0.0 * u, 1e5 * one])


@pytest.mark.parametrize("scheme", [{"kind": "KEP", "order": 2}, {"kind": "KEP", "order": 4},
                                    {"kind": "KEEP", "order": 4},
                                    {"kind": "Hybrid", "central": {"kind": "KEP", "order": 4}}])
@pytest.mark.parametrize("form", ["box", "curvilinear"])
def test_laminar_shear(form, scheme):
    spec, arrays = box_spec((8, 17, 33), (None, None, None), scheme, "none")     # (x nodes are exact)
    if form == "curvilinear":
        X = arrays["nodes_all"]
        s = [2 * np.pi * X[d] / cases.L[d] for d in range(3)]
        arrays["nodes_all"] = X + 0.01 * np.stack([0.0 * X[0], np.sin(s[2]), np.sin(s[1])])
    mesh, sol = cases.build(wmx, spec, arrays)
    _, ref = cases.build(oracle, spec, arrays)
    assert sol.kernel_form() == form
    Q = sol.init_state(shear)
    blk = mesh.blocks[0]
    got = blk.interior(sol.rhs(Q)[0].cpu().numpy())[1]
    want = blk.interior(ref.rhs([q.cpu().numpy() for q in Q])[0])[1]
    assert np.ptp(want, axis=0).max() < 1e-14 * np.abs(want).max() and 1e-5 < np.abs(want).max() < 1e-2
    assert np.abs(got - want).max() <= 1e-12 * np.abs(want).max()
