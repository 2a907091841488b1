"""Rounding of the FP64 right-hand sides: their distance from the oracle evaluated in long double (80
bits) on the same stored nodes and states, as the rms over the block relative to the rms of the
value.  FORMER holds what the kernels that formed every record with divisions, each central flux
with one factor a pair and each cell's sum face by face measured here, with 2% for the last digit
printed: arithmetic that replaces theirs rounds no more."""
import numpy as np
import pytest

import cases
import oracle
import oracle.mesh
from test_gpu_box import HYB, SLIP, box_spec

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("needs a HIP device", allow_module_level=True)
if np.finfo(np.longdouble).nmant < 63:
    pytest.skip("needs a long double of 64 bits", allow_module_level=True)

import wmles_jax_amd as wmx  # noqa: E402

CASES = {"hybrid": ((33, 47, 35), HYB, "vreman"), "kep": ((33, 47, 35), {"kind": "KEP", "order": 4}, "wale"),
         "muscl": ((40, 30, 32), {"kind": "MUSCLHLLC", "limiter": "albada"}, "smagorinsky"),
         "keep": ((40, 30, 32), {"kind": "KEEP", "order": 4}, "none")}
# rho, rho u, rho v, rho w, rho E: mean of three seeds
FORMER = {("box", "hybrid"): (3.33e-15, 1.85e-14, 3.05e-14, 2.97e-14, 3.01e-15),
          ("box", "kep"): (1.39e-15, 2.12e-14, 8.44e-14, 1.04e-13, 1.48e-15),
          ("box", "muscl"): (1.48e-14, 7.80e-15, 7.15e-15, 6.50e-15, 1.29e-14),
          ("box", "keep"): (1.38e-15, 2.84e-14, 5.89e-14, 9.89e-14, 1.48e-15),
          ("curvilinear", "hybrid"): (4.09e-15, 2.14e-14, 3.31e-14, 3.74e-14, 3.82e-15),
          ("curvilinear", "kep"): (2.78e-15, 2.44e-14, 9.15e-14, 1.32e-13, 2.82e-15),
          ("curvilinear", "muscl"): (1.49e-14, 9.33e-15, 8.58e-15, 9.01e-15, 1.30e-14),
          ("curvilinear", "keep"): (2.36e-15, 3.20e-14, 6.48e-14, 1.24e-13, 2.39e-15)}


def in_long_double(solver):
    """The oracle with its metrics formed from the same nodes in long double."""
    for blk in solver.blocks:
        vol, xc, S, xf = oracle.mesh.compute_geometry(np.asarray(blk.X, np.longdouble))
        blk.geom = oracle.mesh.Geom(vol, xc, tuple(S), tuple(xf))
    solver.geoms = tuple(blk.geom for blk in solver.blocks)
    return solver


@pytest.mark.parametrize("form,name", list(FORMER))
def test_right_hand_sides_round_no_more_than_before(form, name):
    n, scheme, sgs = CASES[name]
    spec, arrays = box_spec(n, (None, SLIP, None), scheme, sgs)
    if form == "curvilinear":
        X = arrays["nodes_all"]
        s = [2 * np.pi * X[d] / cases.L[d] for d in range(3)]
        arrays["nodes_all"] = X + 0.02 * min(cases.L) * np.stack(
            [np.sin(s[1]) * np.cos(s[2]), np.sin(s[0]) * np.cos(s[2]), np.cos(s[0]) * np.sin(s[1])])
    mesh, sol = cases.build(wmx, spec, arrays)
    assert sol.kernel_form() == form
    ref = in_long_double(cases.build(oracle, spec, arrays)[1])
    blk, err = mesh.blocks[0], np.zeros(5)
    for seed in range(3):
        Q = cases.interior_noise(mesh.blocks, [np.asarray(q.cpu()) for q in sol.init_state(cases.prim_fn)], seed,
                                 amp=0.05)
        got = blk.interior(sol.rhs(Q)[0].cpu().numpy())
        want = blk.interior(ref.rhs([np.asarray(q, np.longdouble) for q in Q])[0])
        assert want.dtype == np.longdouble
        err += np.sqrt(((got - want) ** 2).mean(axis=(1, 2, 3)) / (want ** 2).mean(axis=(1, 2, 3))).astype(float) / 3
    assert np.all(err <= 1.02 * np.array(FORMER[form, name])), err
