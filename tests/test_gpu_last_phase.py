"""The sweep's last phase inside a step's stages.  Plans of boxes with k walls: the kernels that read the
state take those ghosts from a fill launch, the primitive kernel of the unfused form evaluates them
itself; turning the form over and back keeps the launches and the bits of a plan made that way."""
import pytest

import cases
from test_gpu_box import HYB, SLIP, WM, box_spec, state

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("needs a HIP device", allow_module_level=True)

import wmles_jax_amd as wmx  # noqa: E402


def stepped(s, Q):
    """(fill launches of a step, its state)."""
    s.profile(("fill",))
    out, _ = s.step(Q)
    torch.cuda.synchronize()
    n = s.profile_read().get("fill", (0.0, 0))[1]
    s.profile(())
    return n, out


@pytest.mark.parametrize("walls", [(None, WM, SLIP), (None, WM, None)])
def test_fill_launches_and_bits_of_each_form(walls):
    spec, arrays = box_spec((6, 17, 18), walls, HYB, "vreman")

    def plan(fused):
        mesh, s = cases.build(wmx, spec, arrays, solver_kwargs={"precision": "fp32", "gauge": (1e5, 290.0)})
        s.set_fused_gradients(fused)
        return mesh, s

    mesh, box = plan(True)
    _, split = plan(False)
    Q = state(mesh, box)
    phases = box.fill_phases()[0]
    assert (box.kernel_form(), split.kernel_form()) == ("box", "split")
    n_box, q_box = stepped(box, Q)
    n_split, q_split = stepped(split, Q)
    assert n_split == 3 * (phases - 1)
    assert n_box == 3 * (phases - (walls[2] is None))
    for fused in (False, True, False):
        box.set_fused_gradients(fused)
        n, q = stepped(box, Q)
        assert n == (n_box if fused else n_split)
        assert all(torch.equal(a, b) for a, b in zip(q, q_box if fused else q_split))
