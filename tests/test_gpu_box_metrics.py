"""Boxes whose stored metrics are not exactly products of widths: far from the origin a volume, a
difference of coordinate-sized terms, is off by its rounding.  FP64 right-hand sides stay within the
form's 1e-12 of the oracle, which divides by the stored volume; so do boxes with decreasing axes."""
import numpy as np
import pytest

import cases
import golden_io
import oracle
from test_gpu_box import HYB, WM, box_spec, state

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("needs a HIP device", allow_module_level=True)

import wmles_jax_amd as wmx  # noqa: E402


def rhs_error(arrays, spec):
    mesh, s = cases.build(wmx, spec, arrays)
    _, ref = cases.build(oracle, spec, arrays)
    Q, blk = state(mesh, s), mesh.blocks[0]
    return golden_io.rel_err(blk.interior(s.rhs(Q)[0].cpu().numpy()), blk.interior(ref.rhs(Q)[0]))


@pytest.mark.parametrize("offset", [0.0, 1e2, 1e3, 2.5e3, 1e4, 1e5])
def test_fp64_box_far_from_the_origin(offset):
    spec, arrays = box_spec((9, 17, 18), (None, WM, None), HYB, "vreman")
    arrays["nodes_all"] = arrays["nodes_all"] + offset * np.array(cases.L)[:, None, None, None]
    assert rhs_error(arrays, spec) <= 1e-12


@pytest.mark.parametrize("flip", [(0, 1), (1, 2), (0, 2)])
def test_fp64_box_with_two_decreasing_axes(flip):
    spec, arrays = box_spec((9, 17, 18), (None, WM, None), HYB, "vreman")
    for d in flip:
        arrays["nodes_all"][d] = cases.L[d] - arrays["nodes_all"][d]
    for c in spec["connect"]:
        d = "ijk".index(c[1][0])
        if d in flip:
            c[4][d] = -c[4][d]
    assert rhs_error(arrays, spec) <= 1e-12
