"""Which flux kernel a plan runs: tensor-product blocks the box kernel in both precisions, a block that is
none by one moved node, by curvature, by its order of nodes or (FP64) by the rounding of its volumes
the general one, and one such block sends the whole plan there."""
import numpy as np
import pytest

import cases
from test_gpu_box import HYB, PARAMS, WM, box_spec

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("needs a HIP device", allow_module_level=True)

import wmles_jax_amd as wmx  # noqa: E402

GENERAL = {"fp64": "curvilinear", "fp32": "fused"}


def form(spec, arrays, precision, fused=True):
    s = cases.build(wmx, spec, arrays, solver_kwargs={"precision": precision})[1]
    if not fused:
        s.set_fused_gradients(False)
    return s.kernel_form()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n,walls,scheme,sgs", PARAMS)
def test_tensor_product_blocks_are_boxes(n, walls, scheme, sgs, precision):
    assert form(*box_spec(n, walls, scheme, sgs), precision) == "box"
    assert form(*box_spec(n, walls, scheme, sgs), precision, False) == ("box" if precision == "fp64" else "split")


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_other_blocks_are_not(precision):
    n = (8, 16, 17)
    spec, arrays = box_spec(n, (None, WM, None), HYB, "vreman", move=1e-6)
    assert form(spec, arrays, precision) == GENERAL[precision]
    spec, arrays = box_spec(n, (None, WM, None), HYB, "vreman")
    X = arrays["nodes_all"]
    s = [2 * np.pi * X[d] / cases.L[d] for d in range(3)]
    arrays["nodes_all"] = X + 0.012 * np.stack(
        [np.sin(s[1]) * np.cos(s[2]), np.sin(s[0]) * np.cos(s[2]), np.cos(s[0]) * np.sin(s[1])])
    assert form(spec, arrays, precision) == GENERAL[precision]
    for flip in ((0, 1), (1, 2), (0, 2)):
        spec, arrays = box_spec(n, (None, WM, None), HYB, "vreman")
        for d in flip:
            arrays["nodes_all"][d] = cases.L[d] - arrays["nodes_all"][d]
        for c in spec["connect"]:
            c[4] = [-v if d in flip else v for d, v in enumerate(c[4])]
        assert form(spec, arrays, precision) == GENERAL[precision]
    spec, arrays = cases.multiblock_spec("split", (12, 10, 8), HYB)
    assert form(spec, arrays, precision) == GENERAL[precision]


@pytest.mark.parametrize("offset,fp64", [(1e2, "box"), (1e3, "curvilinear"), (1e5, "curvilinear")])
def test_fp64_boxes_far_from_the_origin_are_not(offset, fp64):
    spec, arrays = box_spec((9, 17, 18), (None, WM, None), HYB, "vreman")
    arrays["nodes_all"] = arrays["nodes_all"] + offset * np.array(cases.L)[:, None, None, None]
    assert form(spec, arrays, "fp64") == fp64


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_one_curved_block_decides_for_the_plan(precision):
    n, L = (12, 10, 8), cases.L
    x, y, z = (np.linspace(0.0, le, k + 1) for le, k in zip(L, n))
    for bend in (0.0, 1e-3):
        X = np.stack(np.meshgrid(x, y, z, indexing="ij"))
        X[1, 7:12] += bend * np.sin(np.pi * X[1, 7:12] / L[1])    # inside the second block only
        spec = {"name": "two", "blocks": ["a", "b"], "ng": 3, "scheme": HYB, "sgs": "vreman",
                "connect": [["a", "imax", "b", "imin", [0.0] * 3], ["b", "imax", "a", "imin", [L[0], 0.0, 0.0]],
                            ["a", "kmin", "a", "kmax", [0.0, 0.0, -L[2]]], ["b", "kmin", "b", "kmax", [0.0, 0.0, -L[2]]]],
                "bcs": [[b, f, dict(WM)] for b in "ab" for f in ("jmin", "jmax")]}
        arrays = {"nodes_a": X[:, :7], "nodes_b": X[:, 6:]}
        assert form(spec, arrays, precision) == ("box" if bend == 0.0 else GENERAL[precision])
