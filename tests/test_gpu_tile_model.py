"""The tile model without a plan answers with what a plan of the same kernel form, precision and blocks
chooses."""
import ctypes as C

import pytest

import cases
from test_gpu_box import HYB, WM, box_spec

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("needs a HIP device", allow_module_level=True)

import wmles_jax_amd as wmx  # noqa: E402
from wmles_jax_amd import _lib  # noqa: E402

FORMS = ("split", "fused", "box", "curvilinear")


@pytest.mark.parametrize("n", [(3, 3, 3), (24, 16, 12), (133, 75, 61)])
@pytest.mark.parametrize("form,precision", [("split", "fp32"), ("fused", "fp32"), ("box", "fp32"), ("box", "fp64"),
                                            ("curvilinear", "fp64")])
def test_the_model_is_the_plans_choice(n, form, precision):
    spec, arrays = box_spec(n, (None, WM, None), HYB, "vreman", move=0.0 if form in ("box", "split") else 1e-3)
    s = cases.build(wmx, spec, arrays, solver_kwargs={"precision": precision})[1]
    s.set_fused_gradients(form != "split")
    assert s.kernel_form() == form
    ci, nt = C.c_int32(), C.c_int32()
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    _lib.check(_lib.lib.wmx_tile_model_form(1, (C.c_int32 * 3)(*n), FORMS.index(form),
                                            _lib.PREC_FP32_BULK if precision == "fp32" else _lib.PREC_FP64, cus,
                                            C.byref(ci), C.byref(nt)))
    assert (ci.value, nt.value) == (s.tiling()[0], s.tiling()[2])
    s.set_tiling(5, 1)
    s.set_tiling(0, 1)
    assert (ci.value, nt.value) == (s.tiling()[0], s.tiling()[2])
