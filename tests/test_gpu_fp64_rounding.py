"""Rounding of the FP64 right-hand sides and steps: their distance from the oracle evaluated in long
double (80 bits) on the same stored nodes and states, as the rms over the block relative to the rms
of the value.  FORMER and FORMER_STEP hold what the kernels measured here that formed every record
with divisions, each central flux with one factor a pair, each cell's sum face by face and each
stage as a0 q0 + a1 (q + dt r), with 2% for the last digit printed: arithmetic that replaces theirs
rounds no more."""
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
# the state after one step of 1e-6 s (rounding of the stages; one seed)
FORMER_STEP = {("box", "hybrid"): (8.137e-17, 7.493e-17, 1.388e-16, 1.083e-16, 5.842e-17),
               ("box", "kep"): (8.144e-17, 7.475e-17, 1.394e-16, 1.085e-16, 5.826e-17),
               ("box", "muscl"): (8.119e-17, 7.457e-17, 1.020e-16, 9.848e-17, 5.774e-17),
               ("box", "keep"): (8.127e-17, 7.481e-17, 1.081e-16, 1.052e-16, 5.822e-17),
               ("curvilinear", "hybrid"): (8.139e-17, 7.553e-17, 1.554e-16, 1.258e-16, 5.808e-17),
               ("curvilinear", "kep"): (8.136e-17, 7.507e-17, 1.559e-16, 1.255e-16, 5.824e-17),
               ("curvilinear", "muscl"): (8.089e-17, 7.515e-17, 1.183e-16, 1.217e-16, 5.790e-17),
               ("curvilinear", "keep"): (8.156e-17, 7.522e-17, 1.192e-16, 1.222e-16, 5.830e-17)}


def in_long_double(solver):
    """The oracle with its metrics formed from the same nodes in long double."""
    for blk in solver.blocks:
        vol, xc, S, xf = oracle.mesh.compute_geometry(np.asarray(blk.X, np.longdouble))
        blk.geom = oracle.mesh.Geom(vol, xc, tuple(S), tuple(xf))
    solver.geoms = tuple(blk.geom for blk in solver.blocks)
    return solver


def build(form, name):
    """(block, solver, long double oracle, noisy state by seed)."""
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
    q0 = [np.asarray(q.cpu()) for q in sol.init_state(cases.prim_fn)]
    return mesh.blocks[0], sol, ref, lambda seed: cases.interior_noise(mesh.blocks, q0, seed, amp=0.05)


def rms_error(got, want):
    assert want.dtype == np.longdouble
    return np.sqrt(((got - want) ** 2).mean(axis=(1, 2, 3)) / (want ** 2).mean(axis=(1, 2, 3))).astype(float)


def wide(Q):
    return [np.asarray(q, np.longdouble) for q in Q]


@pytest.mark.parametrize("form,name", list(FORMER))
def test_right_hand_sides_round_no_more_than_before(form, name):
    blk, sol, ref, noisy = build(form, name)
    err = np.mean([rms_error(blk.interior(sol.rhs(Q)[0].cpu().numpy()), blk.interior(ref.rhs(wide(Q))[0]))
                   for Q in map(noisy, range(3))], axis=0)
    assert np.all(err <= 1.02 * np.array(FORMER[form, name])), err


@pytest.mark.parametrize("form,name", list(FORMER_STEP))
def test_steps_round_no_more_than_before(form, name):
    blk, sol, ref, noisy = build(form, name)
    Q = noisy(0)
    err = rms_error(blk.interior(sol.advance(Q, 1e-6)[0].cpu().numpy()),
                    blk.interior(ref.advance(wide(Q), np.longdouble(1e-6))[0]))
    assert np.all(err <= 1.02 * np.array(FORMER_STEP[form, name])), err
