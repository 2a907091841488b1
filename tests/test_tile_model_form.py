"""Automatic i-planes per tile of each kernel form, against its rule stated here (host only)."""
import ctypes as C

import pytest

_lib = pytest.importorskip("wmles_jax_amd._lib")
SPLIT, FUSED, BOX, CURV = range(4)


def model(dims, form, prec, cus=256):
    ci, nt = C.c_int32(), C.c_int32()
    _lib.check(_lib.lib.wmx_tile_model_form(len(dims) // 3, (C.c_int32 * len(dims))(*dims), form, prec, cus,
                                            C.byref(ci), C.byref(nt)))
    return ci.value, nt.value


def rule(dims, prec, cus=256):
    """Full rounds of 3 (FP32) or 2 workgroups a CU and a remainder, (ci + 1) planes each."""
    part = (0.0, 0.55, 0.78, 1.0) if prec == _lib.PREC_FP32_BULK else (0.0, 0.6, 1.0)
    slots, best = (len(part) - 1) * cus, None
    for ci in range(1, 65):
        T = sum(-(-dims[b] // ci) * -(-dims[b + 1] // 15) * -(-dims[b + 2] // 16) for b in range(0, len(dims), 3))
        cost = (T // slots + part[-(-(T % slots) // cus)]) * (ci + 1)
        if best is None or cost < best[0] - 1e-9:
            best = (cost, ci, T)
    return best[1:]


def test_each_form_answers_with_its_own_rule():
    for dims in ([256, 128, 128], [512, 256, 256], [24, 16, 12], [72, 56, 40, 33, 39, 56], [3, 3, 3], [190, 63, 33]):
        for prec in (_lib.PREC_FP64, _lib.PREC_FP32_BULK):
            assert model(dims, BOX, prec) == rule(dims, prec)
        assert model(dims, CURV, _lib.PREC_FP64) == rule(dims, _lib.PREC_FP64)
        arr, ci, nt = (C.c_int32 * len(dims))(*dims), C.c_int32(), C.c_int32()
        _lib.check(_lib.lib.wmx_tile_model(len(dims) // 3, arr, _lib.PREC_FP32_BULK, 256, C.byref(ci), C.byref(nt)))
        assert model(dims, SPLIT, _lib.PREC_FP32_BULK) == model(dims, FUSED, _lib.PREC_FP32_BULK) == (ci.value, nt.value)
    # the 256 x 128 x 128 box, FP32: 8 planes, three full rounds of 768 workgroups
    assert model([256, 128, 128], BOX, _lib.PREC_FP32_BULK) == (8, 2304)
    with pytest.raises(_lib.WmxError):
        model([3, 3, 3], 4, _lib.PREC_FP64)
