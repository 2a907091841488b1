"""A second workspace bound to a plan: steps captured before it are captured anew, and every form of
the step gives the bits that it gave with the first."""
import ctypes as C

import pytest

import cases
from test_gpu_box import HYB, WM, box_spec, state

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("needs a HIP device", allow_module_level=True)

import wmles_jax_amd as wmx  # noqa: E402
from wmles_jax_amd import _lib  # noqa: E402


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_steps_after_a_second_binding(precision):
    spec, arrays = box_spec((12, 17, 18), (None, WM, None), HYB, "vreman")
    kw = {"precision": precision, **({"gauge": (1e5, 290.0)} if precision == "fp32" else {})}
    mesh, s = cases.build(wmx, spec, arrays, solver_kwargs=kw)
    Q = [torch.as_tensor(q, device="cuda") for q in state(mesh, s)]
    out, dt = [torch.empty_like(q) for q in Q], torch.empty(16, dtype=torch.float64, device="cuda")
    stream = torch.cuda.Stream()

    def step(graph):
        _lib.check(_lib.lib.wmx_step(s._plan, _lib.ptr_array(Q), _lib.ptr_array(out), C.c_void_p(dt.data_ptr()), 0.0,
                                     graph, _lib.stream_ptr(stream)))
        stream.synchronize()
        return [q.clone() for q in out]

    torch.cuda.synchronize()
    want = step(0)
    former = s._ws
    for bound in range(2):
        for graph in (1, 1, 0, 1):
            for q in out:
                q.zero_()
            torch.cuda.synchronize()
            assert all(torch.equal(a, b) for a, b in zip(step(graph), want)), (bound, graph)
        s._ws = torch.empty_like(former)
        torch.cuda.synchronize()
        _lib.check(_lib.lib.wmx_plan_bind_workspace(s._plan, C.c_void_p(s._ws.data_ptr()), s._ws.numel()))
        former.fill_(255)
    if precision == "fp32":
        s.set_persistent(True)
        assert all(torch.equal(a, b) for a, b in zip(step(0), want))
