"""wmx_wall_stats refuses null outputs on the host, as the copies of its former form did: the wall kernel
writes both arrays itself.  A plan without wall-modelled faces has no outputs and takes them."""
import ctypes as C

import pytest

import cases
from test_gpu_box import HYB, NOSLIP, WM, box_spec, state

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("needs a HIP device", allow_module_level=True)

import wmles_jax_amd as wmx  # noqa: E402
from wmles_jax_amd import _lib  # noqa: E402


@pytest.mark.parametrize("wall", [True, False])
def test_null_outputs(wall):
    spec, arrays = box_spec((4, 5, 6), (None, WM if wall else NOSLIP, None), HYB, "vreman")
    mesh, s = cases.build(wmx, spec, arrays)
    Q = [torch.as_tensor(q, device="cuda") for q in state(mesh, s)]
    out = torch.full((2, 2 * 4 * 6), -1.0, dtype=torch.float64, device="cuda")
    both = [C.c_void_p(out[k].data_ptr()) for k in range(2)]
    for tau, qw in ((both[0], None), (None, both[1]), (None, None)):
        assert (_lib.lib.wmx_wall_stats(s._plan, _lib.ptr_array(Q), tau, qw, _lib.stream_ptr()) != 0) == wall
    torch.cuda.synchronize()
    assert bool((out == -1.0).all())
    _lib.check(_lib.lib.wmx_wall_stats(s._plan, _lib.ptr_array(Q), *both, _lib.stream_ptr()))
    torch.cuda.synchronize()
    assert bool((out[0] > 0.0).all()) == wall
