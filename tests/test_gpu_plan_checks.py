"""Plans that are refused: each with its status, before anything is computed from the
segment that is wrong (a window of 2^29 and more cells once kept the upload counting)."""
import ctypes as C

import pytest

import openpstd_amd as P  # noqa: F401 (loads the library)
from openpstd_amd import abi_types as T
from openpstd_amd._lib import lib

pytestmark = pytest.mark.gpu
INT_MAX, INT_MIN = 2**31 - 1, -2**31


class Domain(C.Structure):
    _fields_ = [("nx", C.c_int32), ("ny", C.c_int32), ("rho", C.c_float), ("is_pml", C.c_int32), ("is_rigid", C.c_int32),
                ("pml_px", C.c_void_p), ("pml_py", C.c_void_p), ("pml_vx", C.c_void_p), ("pml_vy", C.c_void_p)]


class Plan(C.Structure):
    _fields_ = [("n_domains", C.c_int32), ("domains", C.POINTER(Domain)),
                ("n_segments", C.c_int32), ("segments", C.POINTER(T.pstd_plan_segment)),
                ("n_receivers", C.c_int32), ("receivers", C.c_void_p),
                ("dx", C.c_float), ("dt", C.c_float), ("c1", C.c_float), ("patch_error", C.c_float),
                ("rk_alpha", C.c_float * 6)]


def upload(**wrong):
    dom = (Domain * 1)(Domain(nx=100, ny=90, rho=1.2))
    seg = (T.pstd_plan_segment * 2)()
    for s in seg:
        for name, v in dict(domain=0, direction=0, field=0, line_begin=0, line_end=90, side1=-1, side2=-1, wlen=32,
                            table_len=256, c_main1=1.0, c_main2=1.0).items():
            setattr(s, name, v)
    for name, v in wrong.items():  # (the second segment: the first one is sound)
        setattr(seg[1], name, v)
    plan = Plan(n_domains=1, domains=dom, n_segments=2, segments=seg, dx=0.2, dt=1e-4, c1=340.0, patch_error=70.0)
    ctx = C.c_void_p()
    assert lib().pstd_ctx_create(0, C.byref(ctx)) == T.PSTD_OK
    try:
        return lib().pstd_ctx_upload_plan(ctx, C.byref(plan)), lib().pstd_ctx_last_error(ctx).decode()
    finally:
        lib().pstd_ctx_destroy(ctx)


def test_the_plan_itself_is_accepted():
    assert upload() == (T.PSTD_OK, "")


@pytest.mark.parametrize("wlen", [33, 2**20, 2**29 - 50, 2**29, 2**29 + 1, 2**30 - 51, 2**30 - 50, 2**30, INT_MAX])
def test_windows_above_32_are_refused(wlen):
    rc, err = upload(wlen=wlen)
    assert rc == T.PSTD_ERR_UNSUPPORTED and "window half-length %d above 32" % wlen in err


@pytest.mark.parametrize("wrong", [
    dict(wlen=0), dict(wlen=INT_MIN), dict(domain=-1), dict(domain=1), dict(side1=1), dict(side2=INT_MAX), dict(direction=2),
    dict(field=-1), dict(line_begin=-1), dict(line_end=91), dict(line_end=0), dict(line_begin=INT_MIN, line_end=INT_MAX),
    dict(line_begin=INT_MAX, line_end=INT_MIN), dict(table_len=128), dict(table_len=300), dict(side1=0, side1_offset=1)])
def test_invalid_segments_are_refused(wrong):
    rc, err = upload(**wrong)
    assert rc == T.PSTD_ERR_INVALID and err
