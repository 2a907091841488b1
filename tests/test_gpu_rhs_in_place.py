"""wmx_rhs and wmx_rhs_filled with r == q, and with the blocks' outputs on each other's inputs: the same
bits as with separate buffers, in both precisions, on boxes and curvilinear blocks."""
import numpy as np
import pytest

import cases
from test_gpu_box import HYB, WM, box_spec

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("needs a HIP device", allow_module_level=True)

import wmles_jax_amd as wmx  # noqa: E402
from wmles_jax_amd import _lib  # noqa: E402


def solver(kind, precision):
    kw = {"precision": precision, **({"gauge": (1e5, 290.0)} if precision == "fp32" else {})}
    if kind == "two blocks":
        spec, arrays = cases.multiblock_spec("split", (12, 17, 18), HYB)
    else:
        spec, arrays = box_spec((20, 33, 34), (None, WM, None), HYB, "vreman")
        if kind == "curvilinear":
            X, turn = arrays["nodes_all"], [1, 2, 0]
            period = np.array(cases.L)[turn, None, None, None]
            arrays["nodes_all"] = X + 0.01 * np.sin(2 * np.pi * X[turn] / period)
    return cases.build(wmx, spec, arrays, solver_kwargs=kw)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("kind", ["box", "curvilinear", "two blocks"])
def test_rhs_in_place(kind, precision):
    mesh, s = solver(kind, precision)
    Q = s.apply_bcs([torch.as_tensor(q, device="cuda") for q in cases.interior_noise(
        mesh.blocks, [np.asarray(q.cpu()) for q in s.init_state(cases.prim_fn)], 3, amp=0.05)])
    want = s.rhs(Q)
    stream = _lib.stream_ptr()
    for swap in ([False, True] if len(Q) == 2 and Q[0].shape == Q[1].shape else [False]):
        for filled in (False, True):
            work = [q.clone() for q in Q]
            out = work[::-1] if swap else work
            rc = (_lib.lib.wmx_rhs_filled(s._plan, _lib.ptr_array(work), _lib.ptr_array(out), stream) if filled
                  else _lib.lib.wmx_rhs(s._plan, _lib.ptr_array(work), _lib.ptr_array(out), 0.0, stream))
            _lib.check(rc)
            assert all(torch.equal(a, b) for a, b in zip(out, want)), (swap, filled)
