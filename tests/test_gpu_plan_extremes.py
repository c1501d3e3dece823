"""Plans whose sizes and offsets overflow 32 or 64 bits are refused like any other that
does not fit: domains near the largest extents, neighbour offsets near the ends of
their type, a negative number of domains."""
import ctypes as C

import pytest

from openpstd_amd import abi_types as T
from openpstd_amd._lib import lib

from test_gpu_plan_checks import INT_MAX, INT_MIN, Domain, Plan

pytestmark = pytest.mark.gpu


def upload(nx=100, ny=90, n_domains=2, **segment):
    dom = (Domain * 2)(Domain(nx=100, ny=90, rho=1.2), Domain(nx=nx, ny=ny, rho=1.2))
    seg = (T.pstd_plan_segment * 1)()
    for name, v in dict(dict(domain=0, line_end=90, side1=-1, side2=-1, wlen=32, table_len=256, c_main1=1.0,
                             c_main2=1.0), **segment).items():
        setattr(seg[0], name, v)
    plan = Plan(n_domains=n_domains, domains=dom, n_segments=1, segments=seg, dx=0.2, dt=1e-4, c1=340.0, patch_error=70.0)
    ctx = C.c_void_p()
    assert lib().pstd_ctx_create(0, C.byref(ctx)) == T.PSTD_OK
    try:
        return lib().pstd_ctx_upload_plan(ctx, C.byref(plan)), lib().pstd_ctx_last_error(ctx).decode()
    finally:
        lib().pstd_ctx_destroy(ctx)


def test_the_plan_itself_is_accepted():
    assert upload(side1=1, side2=1) == (T.PSTD_OK, "")


@pytest.mark.parametrize("nx, ny", [(INT_MAX, INT_MAX), (2**31 - 2**16, 2**31 - 2**17), (2**30, 2**30), (2**16, 2**16),
                                    (INT_MAX, 1), (1, INT_MAX), (2**27, 1), (11586, 11585)])
def test_domains_above_a_block_are_refused(nx, ny):
    rc, err = upload(nx, ny)
    assert rc == T.PSTD_ERR_UNSUPPORTED and "domain of %d cells" % (nx * ny) in err


@pytest.mark.parametrize("offset", [1, -1, INT_MAX, INT_MAX - 89, INT_MAX - 90, INT_MIN, INT_MIN + 90])
@pytest.mark.parametrize("side", ["side1", "side2"])
def test_neighbour_lines_outside_the_neighbour_are_refused(side, offset):
    rc, err = upload(**{side: 1, side + "_offset": offset})
    assert rc == T.PSTD_ERR_INVALID and "outside its neighbour" in err


def test_a_negative_number_of_domains_is_refused():
    for n in (-1, INT_MIN):
        rc, err = upload(n_domains=n)
        assert rc == T.PSTD_ERR_INVALID and "number of domains" in err
