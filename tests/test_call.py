"""The compiled call path takes, refuses and raises what the ctypes path it stands in for does."""
import ctypes

import pytest


class Holder:
    def __init__(self, p):
        self.p = p

    def data_ptr(self):
        return self.p


@pytest.mark.parametrize("args", [
    (None, None, None, 0, None), (None, None, None, -1, None), (None, None, None, 4, None), (None, None, None, True, None),
    (0, 0, 0, 1 << 32, 0), (None, None, None, -(1 << 40), None), (Holder(0), Holder(16), None, 0, 0), (Holder(None), None, None, 0, None),
    (None, None, None, ctypes.c_int(0), None), (ctypes.c_void_p(0), None, None, 0, None),
    (None, None, None, 0, None, 7), (None, None, None, 0), (None, None, None, 0.0, None), (object(), None, None, 0, None), (Holder("x"), None, None, 0, 1.5),
])
def test_same_answer_as_ctypes(cf, args):
    def outcome(call):
        try:
            return call(*args)
        except Exception as e:
            return type(e), getattr(e, "code", None)

    assert outcome(cf.cf_swiglu_forward) == outcome(cf._checked("cf_swiglu_forward", cf.raw_cf_swiglu_forward))


def test_floats_sizes_and_outputs(cf):
    n, m = ctypes.c_size_t(7), ctypes.c_size_t(7)
    assert cf.cf_moe_grouped_gelu_workspace_bytes(16, 96, 8, 2048, 1408, ctypes.byref(n)) is None
    assert cf.raw_cf_moe_grouped_gelu_workspace_bytes(16, 96, 8, 2048, 1408, ctypes.byref(m)) == 0 and n.value == m.value > 7
    for value in (448.0, 448, -1, 0.0):          # a float parameter; a null output is refused whatever it is
        with pytest.raises(type(cf)._failed.__globals__["CfError"]):
            cf.cf_fp8_scale_from_amax(None, value, None, None, None)
    assert cf.cf_fp8_quantize_e4m3.__name__ == "cf_fp8_quantize_e4m3"
