"""Box ranges, occupied lists, target flags and class lists of all levels at
once (wbfmm_hip_tree_levels, wbfmm_hip_tree_targets) against numpy: levels
below one wavefront, one chunk and many chunks of boxes, few and many points,
points in one corner, no target that is not a source's box, no target."""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

_vp = ctypes.c_void_p


def codes_of(rng, n, spread):
    x = (rng.uniform(0, 1, (n, 3)) ** spread * 2 ** 20).astype(np.uint64)
    code = np.zeros(n, np.uint64)
    for b in range(20):
        for a in range(3):
            code |= ((x[:, a] >> np.uint64(b)) & np.uint64(1)) << np.uint64(3 * b + a)
    return np.sort(code)


@pytest.mark.parametrize("n,nt,hi,spread", [(1, 1, 3, 1), (2, 0, 2, 1), (255, 300, 4, 1),
                                            (5000, 4097, 5, 3), (70000, 1, 6, 1),
                                            (0, 5, 3, 1)])
def test_levels_and_targets(wb, n, nt, hi, spread):
    lib = wb.lib()
    rng = np.random.default_rng(7 * n + nt)
    src, tgt = codes_of(rng, n, spread), codes_of(rng, nt, 1)
    up = lambda a: wb.DeviceBuffer.from_array(a if a.size else np.zeros(1, a.dtype))
    d_src, d_tgt, d_tot = up(src), up(tgt), wb.DeviceBuffer(4 * 170)
    bufs = {k: [wb.DeviceBuffer(4 * 8 ** l) for l in range(hi + 1)]
            for k in ("start", "end", "occ", "flag", "act", "cls")}
    arr = lambda k: (_vp * 17)(*[b.ptr for b in bufs[k]])
    # the levels in two calls, as refine and a later refine would
    for lo, h in ((0, hi - 1), (hi, hi)):
        assert lib.wbfmm_hip_tree_levels(_vp(d_src.ptr), n, lo, h, arr("start"), arr("end"),
                                         arr("occ"), _vp(d_tot.ptr)) == 0
    assert lib.wbfmm_hip_tree_targets(_vp(d_tgt.ptr), nt, hi, arr("start"), arr("end"),
                                      arr("flag"), arr("act"), arr("cls"), _vp(d_tot.ptr)) == 0
    wb.sync()
    tot = d_tot.download(np.zeros(170, np.uint32)).reshape(17, 10)
    for l in range(hi + 1):
        nb = 8 ** l
        get = lambda k: bufs[k][l].download(np.zeros(nb, np.uint32))
        box = (src >> np.uint64(3 * (20 - l))).astype(np.int64)
        cnt = np.bincount(box, minlength=nb)
        first = np.concatenate([[0], np.cumsum(cnt)[:-1]])
        assert np.array_equal(get("start"), np.where(cnt > 0, first, 0)), l
        assert np.array_equal(get("end"), np.where(cnt > 0, first + cnt, 0)), l
        occ = np.flatnonzero(cnt)
        assert tot[l, 0] == len(occ) and np.array_equal(get("occ")[:len(occ)], occ), l
        on = cnt > 0
        on[(tgt >> np.uint64(3 * (20 - l))).astype(np.int64)] = True
        act = np.flatnonzero(on)
        assert np.array_equal(get("flag"), on), l
        assert tot[l, 1] == len(act) and np.array_equal(get("act")[:len(act)], act), l
        assert np.array_equal(tot[l, 2:], np.bincount(act & 7, minlength=8)), l
        assert np.array_equal(get("cls")[:len(act)], act[np.argsort(act & 7, kind="stable")]), l
    for b in [d_src, d_tgt, d_tot] + sum(bufs.values(), []):
        b.free()


def test_all_classes(wb):
    lib = wb.lib()
    for l in (1, 2, 5):
        b = wb.DeviceBuffer(4 * 8 ** l)
        assert lib.wbfmm_hip_all_classes(l, _vp(b.ptr)) == 0
        k = np.arange(8 ** l)
        assert np.array_equal(b.download(np.zeros(8 ** l, np.uint32)),
                              k[np.argsort(k & 7, kind="stable")])
        b.free()
    assert lib.wbfmm_hip_all_classes(0, None) != 0 and lib.wbfmm_hip_all_classes(11, None) != 0


def test_points_sorted(wb):
    # device and strided host points, ties (of the codes without their low
    # bits) kept in the caller's order, the count of points outside
    lib = wb.lib()
    rng = np.random.default_rng(3)
    for n, stride, low in ((1, 24, 0), (1000, 40, 0), (5000, 24, 0), (5000, 24, 45), (9, 24, 57)):
        x = rng.uniform(0.01, 0.99, (n, stride // 8))
        x[n // 2:, :3] = x[:n - n // 2, :3]
        if n == 1000:
            x[7, 1] = 1.5
        raw, xyz = wb.DeviceBuffer(32 * n), wb.DeviceBuffer(32 * n)
        codes, idx = wb.DeviceBuffer(8 * n), wb.DeviceBuffer(4 * n)
        x0 = np.zeros(3)
        for dev in (False, True):
            src = wb.DeviceBuffer.from_array(x) if dev else None
            nbad = ctypes.c_uint(99)
            assert lib.wbfmm_hip_points_sorted(
                _vp(src.ptr if dev else x.ctypes.data), ctypes.c_size_t(stride), n,
                _vp(x0.ctypes.data), ctypes.c_double(1.0), low, _vp(raw.ptr), _vp(xyz.ptr),
                _vp(codes.ptr), _vp(idx.ptr), ctypes.byref(nbad)) == 0
            assert nbad.value == (1 if n == 1000 else 0)
            i = idx.download(np.zeros(n, np.uint32))
            c = codes.download(np.zeros(n, np.uint64))
            g = (x[:, :3] * 2 ** 20).astype(np.uint64)
            want = np.zeros(n, np.uint64)
            for b in range(21):
                for a in range(3):
                    want |= ((g[:, a] >> np.uint64(b)) & np.uint64(1)) << np.uint64(3 * b + a)
            if n != 1000:
                order = np.argsort(want >> np.uint64(low), kind="stable")
                assert np.array_equal(i, order) and np.array_equal(c, want[order])
                assert np.array_equal(xyz.download(np.zeros((n, 4)))[:, :3], x[order, :3])
            if src:
                src.free()
        for b in (raw, xyz, codes, idx):
            b.free()
