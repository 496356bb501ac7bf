"""The kernels' exponentials and activations equal their plain forms for every
one of the 2^32 floats (infinities, NaN and subnormals among them), in waves of
ordinary arguments and in waves that mix them with special ones; and the plain
forms are the CPU oracle's."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FORMS = ["expf_", "expf_br", "exp2_neg", "sigmoid", "sigmoid_br", "softplus", "softplus_br", "silu",
         "gelu", "gelu_br", "gelu_hw"]


@pytest.fixture(scope="module")
def lib():
    here = os.path.dirname(os.path.abspath(__file__))
    so = os.path.join(here, "libmath_forms.so")
    if not os.path.exists(so):
        subprocess.run(["make", "-s", "-C", here], check=True)
    return ctypes.CDLL(so)


@pytest.mark.parametrize("scatter", [0, 1])
@pytest.mark.parametrize("form", FORMS)
def test_every_float(lib, form, scatter):
    res = (ctypes.c_ulonglong * 2)()
    assert lib.math_forms_check(FORMS.index(form), scatter, res) == 0
    assert res[0] == 0, f"{res[0]} floats differ, the last 0x{res[1]:08x}"


@pytest.mark.parametrize("form,ref", [("expf_", "ref_expf"), ("exp2_neg", "ref_exp2_neg"),
                                      ("softplus", "ref_softplus"), ("silu", "ref_silu"),
                                      ("gelu", "ref_gelu")])
def test_plain_forms_are_the_oracles(lib, oracle, form, ref):
    step, n = 65521, 65536  # odd: every exponent and many mantissas
    got = np.zeros(n, np.float32)
    assert lib.math_forms_plain(FORMS.index(form), ctypes.c_uint32(step), n,
                                got.ctypes.data_as(ctypes.c_void_p)) == 0
    x = (np.arange(n, dtype=np.uint64) * step).astype(np.uint32).view(np.float32)
    f = getattr(oracle.lib(), ref)
    want = np.array([f(ctypes.c_float(v)) for v in x], np.float32)
    same = (got.view(np.uint32) == want.view(np.uint32)) | (np.isnan(got) & np.isnan(want))
    assert same.all(), x[~same][:5]
