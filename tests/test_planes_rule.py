"""Which launches the bit-plane channel sum takes (dd_tdd_planes_pay, host only)."""
import ctypes as C

import pytest


@pytest.fixture
def pays(dd):
    fn = dd.lib().dd_tdd_planes_pay
    fn.restype = C.c_int
    fn.argtypes = [C.c_uint] + [C.c_size_t] * 5
    return lambda nbits, nch, nout, ndm, step=2: bool(fn(nbits, nch, -(-nout // 4096), nout, ndm, int(15 * step)))


# times on the other kernels and on bit planes (us)
@pytest.mark.parametrize("nbits,nch,nout,ndm,other,planes", [
    (4, 16, 6144, 2560, 41, 61), (4, 32, 8192, 1536, 44, 58), (4, 64, 6554, 1024, 62.2, 69.5),
    (4, 16, 98559, 1454, 208, 284), (4, 32, 7877, 13432, 180, 208),
    (4, 64, 9600, 1024, 66.5, 70.4), (4, 64, 26214, 256, 63.8, 69.1), (4, 64, 6144, 2560, 64, 80),
    (8, 32, 6144, 2080, 49, 69), (8, 64, 8192 * 4, 520, 74, 87), (8, 64, 6144, 4096, 116, 144),
    (8, 256, 6144, 2080, 186, 237), (8, 256, 9600, 1024, 160.4, 173.7), (8, 1024, 6144, 2080, 709, 806),
])
def test_launches_that_bit_planes_slow_down_stay_off_them(pays, nbits, nch, nout, ndm, other, planes):
    assert other < planes and not pays(nbits, nch, nout, ndm)


@pytest.mark.parametrize("nbits,nch,nout,ndm,other,planes", [
    (4, 64, 65536, 448, 90, 69), (4, 256, 65536, 384, 311, 209), (4, 1024, 32768, 384, 416, 329),
    (4, 1024, 999178, 1167, 22900, 14600), (8, 256, 32768, 1024, 346, 289),
    (8, 1024, 15625, 3000, 1920, 1430), (8, 1024, 26214, 256, 447.3, 371.5), (8, 1024, 65536, 1024, 2521, 1946),
    (2, 64, 8192, 768, 72, 49), (2, 512, 4 * 600000, 1024, 21800, 8300), (1, 64, 6144, 1024, 74, 43),
    (1, 512, 176150, 501, 990, 350),
])
def test_launches_that_bit_planes_speed_up_take_them(pays, nbits, nch, nout, ndm, other, planes):
    assert planes < other and pays(nbits, nch, nout, ndm)


# delays step samples apart from DM to DM
@pytest.mark.parametrize("nch,nout,ndm,step,other,planes", [
    (512, 109686, 58, 255.6, 401, 201), (512, 4460, 939, 323.0, 511, 230), (1000, 89900, 81, 163.6, 644, 330),
    (328, 99619, 184, 88.3, 252, 194), (200, 65470, 91, 75.5, 110, 87), (512, 11420, 491, 124.2, 266, 173),
    (200, 8237, 2422, 165.1, 195, 292), (200, 12397, 2361, 169.4, 302, 352), (96, 83165, 1190, 256.5, 495, 527),
    (200, 47188, 2296, 157.4, 808, 877),
])
def test_wide_windows(pays, nch, nout, ndm, step, other, planes):
    """1 DM per wave, and one workgroup per CU, where the windows need it."""
    assert pays(4, nch, nout, ndm, step) == (planes < other)


@pytest.mark.parametrize("nbits", [1, 2, 4, 8, 16, 32])
def test_smallest_launches_and_wide_samples(pays, nbits):
    assert not pays(nbits, 64, 1, 1) and not pays(nbits, 1024, 4096, 16)
    if nbits > 8:
        assert not pays(nbits, 1024, 1 << 20, 2048)


@pytest.mark.parametrize("nbits,planes", [(1, 2), (2, 2), (4, 2), (8, 1)])
def test_tilings_are_counted_as_they_are_listed(dd, nbits, planes):
    """Without a buffer, with one too short and with one that holds them all."""
    for name in ("dd_tdd_planes_tilings", "dd_tdd_lds_tilings"):
        fn = getattr(dd.lib(), name)
        fn.restype, fn.argtypes = C.c_int, [C.c_uint, C.c_void_p, C.c_int]
        buf = (C.c_uint * (5 * 64))()
        n = fn(nbits, buf, 64)
        assert fn(nbits, None, 0) == n and fn(nbits, (C.c_uint * 5)(), 1) == n
        shapes = [tuple(buf[5 * i : 5 * i + 4]) for i in range(n)]
        assert len(set(shapes)) == n and sum(s[0] == 64 and s[2] == 8 for s in shapes) >= planes
        if name == "dd_tdd_planes_tilings":
            assert n == planes
