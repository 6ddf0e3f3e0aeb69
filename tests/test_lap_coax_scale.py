"""The Laplace coaxial tables of any width from those of width 1: the powers
of the width against the tables of width 2 (exact), and the scaled tables
against the host's."""

import ctypes

import numpy as np
import pytest

_vp = ctypes.c_void_p
ORDERS = [2, 3, 9, 12, 16, 20, 24]


def host_table(wb, P, kind, w):
    lib = wb.lib()
    A2 = np.zeros(((P.NR if kind == 2 else 1), P.KT * 64))
    p, a = ctypes.byref(P), A2.ctypes.data_as(_vp)
    rc = (lib.wbfmm_hip_lap_m2l_coax(p, ctypes.c_double(w), a) if kind == 2 else
          lib.wbfmm_hip_lap_shift_coax(p, kind, ctypes.c_double(w), a))
    assert rc == 0
    return A2


def plan(wb, N):
    P = wb.M2LPlan()
    assert wb.lib().wbfmm_hip_lap_m2l_tables(N, ctypes.byref(P), None, None, None) == 0
    return P


def powers(wb, P, kind):
    e = np.zeros(P.KT * 64, np.int8)
    assert wb.lib().wbfmm_hip_lap_coax_powers(ctypes.byref(P), kind, e.ctypes.data_as(_vp)) == 0
    return e


@pytest.mark.parametrize("kind", [0, 1, 2])
@pytest.mark.parametrize("N", ORDERS)
def test_powers(N, kind):
    import wbfmm_amd as wb
    P = plan(wb, N)
    one, two = host_table(wb, P, kind, 1.0), host_table(wb, P, kind, 2.0)
    e = powers(wb, P, kind).astype(int)
    # pow(2 r, k) and 2^k pow(r, k): one rounding of the last place apart
    assert np.abs(np.ldexp(one, e) - two).max(initial=0) <= 0 or np.all(
        np.abs(np.ldexp(one, e) - two) <= 2 ** -52 * np.abs(two))


@pytest.mark.gpu
@pytest.mark.parametrize("w", [1.0, 0.3, 1.7e-3, 4.92e-7])
@pytest.mark.parametrize("kind", [0, 1, 2])
@pytest.mark.parametrize("N", ORDERS)
def test_scaled(wb, N, kind, w):
    lib = wb.lib()
    P = plan(wb, N)
    one, want = host_table(wb, P, kind, 1.0), host_table(wb, P, kind, w)
    e = powers(wb, P, kind)
    d1, de, do = (wb.DeviceBuffer.from_array(one), wb.DeviceBuffer.from_array(e),
                  wb.DeviceBuffer(one.nbytes))
    sz = ctypes.c_size_t
    assert lib.wbfmm_hip_lap_coax_scale(_vp(d1.ptr), _vp(de.ptr), sz(one.size), sz(e.size),
                                        ctypes.c_double(w), _vp(do.ptr)) == 0
    got = do.download(np.zeros_like(one))
    # (4.92e-7: the last entries of order 24 are near the largest double, and
    # w^-49 is beyond it)
    assert np.isfinite(want).all()
    # the host's rounding of r w, taken to a power of up to 2 N + 1, and one
    # rounding each of two powers and two products
    assert np.all(np.abs(got - want) <= (2 * N + 6) * 2 ** -53 * np.abs(want))
