"""CFL step of a box block where a cell's pressure is zero or nearly zero to rounding: the cells that
the first pass may leave out must not include one whose exact step is no number or the smallest."""
import numpy as np
import pytest

import cases
import oracle
from test_gpu_box import HYB, WM, box_spec, state

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("needs a HIP device", allow_module_level=True)

import wmles_jax_amd as wmx  # noqa: E402


def pair(n):
    spec, arrays = box_spec(n, (None, WM, None), HYB, "vreman")
    mesh, s = cases.build(wmx, spec, arrays)
    return mesh.blocks[0], s, cases.build(oracle, spec, arrays)[1], state(mesh, s)[0]


def kinetic(q, reciprocal):
    """rho |u|^2 / 2 with the velocities as quotients or as products with 1 / rho."""
    v = [q[1 + c] * (1.0 / q[0]) if reciprocal else q[1 + c] / q[0] for c in range(3)]
    return (0.5 * q[0]) * ((v[0] * v[0] + v[1] * v[1]) + v[2] * v[2])


@pytest.mark.parametrize("ulps", [1, 2])
def test_pressure_below_zero_by_rounding_is_no_number(ulps):
    blk, s, ref, base = pair((8, 16, 8))
    rng = np.random.default_rng(ulps)
    q = np.stack([rng.uniform(0.5, 2.0, 200000), *(rng.uniform(-80.0, 80.0, (3, 200000)))])
    E = kinetic(q, False)
    for _ in range(ulps):
        E = np.nextafter(E, 0.0)
    at = np.flatnonzero(E - kinetic(q, True) > 0.0)[:40]         # the two forms disagree on the sign
    assert len(at) == 40 and np.all(E[at] - kinetic(q, False)[at] < 0.0)
    for i in at:
        Q = base.copy()
        blk.interior(Q)[:, 3, 7, 5] = [*q[:, i], E[i]]
        with np.errstate(all="ignore"):
            assert np.isnan(float(np.asarray(ref.max_dt([Q]))))
        assert np.isnan(float(s.max_dt([Q])))
        assert np.isnan(float(s.step([Q])[1]))


@pytest.mark.parametrize("n", [(8, 16, 8), (11, 31, 13)])
def test_fast_cells_of_small_pressure_decide_as_the_oracle_says(n):
    """Two equally fast cells of a workgroup whose pressures are fractions of their total energy."""
    blk, s, ref, base = pair(n)
    for frac in 10.0 ** np.arange(-16.0, 0.0, 0.5):
        Q = base.copy()
        for k, (at, u) in enumerate((((0, 0, 0), 3.0e4), ((-1, -1, -1), -3.0e4))):
            m = [1.1 + 0.1 * k, 0.0, 0.0, 0.0]
            m[1:] = m[0] * np.array([u, 0.3 * u, -0.2 * u])
            blk.interior(Q)[(slice(None),) + at] = [*m, kinetic(np.array(m), False) / (1.0 - frac)]
        want, got = float(np.asarray(ref.max_dt([Q]))), float(s.max_dt([Q]))
        assert (np.isnan(got) and np.isnan(want)) or abs(got - want) <= 1e-13 * want, (frac, got, want)
