"""The VALU issue ceiling of calib.hip is one: no kernel issues faster.  The
1080p, 1 M-triangle frame's shading issues 651 G wavefront instructions/s."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu


def test_valu_ceiling(gpu_ctx):
    from openclrenderer_amd import build as b
    cal = C.CDLL(b.CALIB_LIB)
    cal.ocr_calib_valu.argtypes = [C.c_int, C.c_uint32]
    cal.ocr_calib_valu.restype = C.c_double
    f32, f64 = cal.ocr_calib_valu(0, 1024), cal.ocr_calib_valu(1, 1024)
    print(f32, f64)
    assert f32 > 700e9 and 0 < f64 < f32
