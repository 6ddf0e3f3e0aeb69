"""A tree used again clears its level arrays by the boxes that were written
(wbfmm_hip_clear_rows): every level of the second and third solve must hold
what a fresh tree of the same points holds, and zeros in every other box."""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def sphere(rng, n, cap):
    """n points on the unit sphere, z above or below as cap says"""
    x = rng.normal(size=(n, 3))
    x /= np.linalg.norm(x, axis=1)[:, None]
    if cap:
        x[:, 2] = cap * np.abs(x[:, 2])
    return np.ascontiguousarray(x)


@pytest.mark.parametrize("kind", ["laplace", "fp32", "vector", "helmholtz", "mixed"])
def test_reused_tree(wb, kind):
    rng = np.random.default_rng(3)
    n, depth, p = 700, 4, 6
    helm, nq = kind in ("helmholtz", "mixed"), 3 if kind == "vector" else 1
    bits = 32 if kind in ("fp32", "mixed") else 64
    orders = [0, p] + [p] * (depth - 1)
    x0, D = np.array([-1.1, -1.1, -1.1]), 2.2
    q = rng.normal(size=(n, 2 if helm else nq))

    def solver(xs, xt):
        if helm:
            return wb.HelmholtzSolver(xs, x0, D, depth, orders, orders, 2.0, targets=xt,
                                      precision=bits)
        return wb.LaplaceSolver(xs, x0, D, depth, orders, orders, targets=xt, precision=bits,
                                host_mirror=False, nq=nq)

    def levels(s):
        return [s.coefficients(l, w) for l in range(2, depth + 1) for w in (0, 1)]

    # above, below, everywhere; registered targets, then none
    sets = [(sphere(rng, n, c), t) for c, t in ((1, 1), (-1, 1), (0, 1), (1, 0), (-1, 1))]
    used = solver(sets[0][0], sets[0][0])
    for xs, with_targets in sets:
        xt = sphere(rng, n, 0)[:300] if with_targets else None
        used.xs, used.targets, used.ntgt = xs, xt, 300
        fresh = solver(xs, xt)
        for s in (used, fresh):
            s.build_tree()
            s.passes(q, sstr=q.shape[1])
            s.passes(q, sstr=q.shape[1])   # (clears whole levels first)
        for a, b in zip(levels(used), levels(fresh)):
            assert np.abs(b).max() > 0
            assert np.array_equal(a, b)
        # the same points again: levels cleared by the lists of the first time
        used.build_tree()
        used.passes(q, sstr=q.shape[1])
        for a, b in zip(levels(used), levels(fresh)):
            assert np.array_equal(a, b)
        fresh.close()
    used.close()


@pytest.mark.parametrize("kind", ["laplace", "fp32", "helmholtz", "mixed"])
def test_levels_that_the_caller_wrote(wb, kind):
    """t->mps and t->mpr are public: what a caller stored there is cleared by
    coefficient_init, and by leaf_expansions with zero_expansions, whether the
    library last left the array zeroed or written by its passes"""
    rng = np.random.default_rng(4)
    n, depth, p, k = 500, 3, 5, 2.0
    helm = kind in ("helmholtz", "mixed")
    orders = [0, p] + [p] * (depth - 1)
    x0, D = np.array([-1.1, -1.1, -1.1]), 2.2
    xs, q = sphere(rng, n, 0), rng.normal(size=(n, 2 if helm else 1))
    make = wb.HelmholtzSolver if helm else wb.LaplaceSolver
    args = (xs, x0, D, depth, orders, orders) + ((k,) if helm else ())
    s = make(*args, targets=xs, precision=32 if kind in ("fp32", "mixed") else 64,
             **({} if helm else {"host_mirror": False}))
    L = wb.lib()

    def levels():
        return [s.coefficients(l, w) for l in range(2, depth + 1) for w in (0, 1)]

    def scribble(which):
        """every coefficient of the levels something else, as a caller does"""
        es = 4 if kind in ("fp32", "mixed") else 8
        for l in range(2, depth + 1):
            a = (s.tree.contents.mps, s.tree.contents.mpr)[which][l]
            nbytes = 8 ** l * (p + 1) ** 2 * es * (2 if helm else 1)
            assert L.wbfmm_hip_memset(a, 0x3f, nbytes) == 0

    s.build_tree()
    s.passes(q)
    want = levels()
    for after_passes in (False, True):
        for which in (0, 1):
            s.build_tree()
            if after_passes:
                s.passes(q)
            scribble(which)
            s.build_tree()
            assert all(not a.any() for a in levels())
            s.passes(q)
            assert all(np.array_equal(a, b) for a, b in zip(levels(), want))
    # the leaf level alone, by zero_expansions
    s.build_tree()
    L.wbfmm_hip_memset(s.tree.contents.mps[depth], 0x3f, 8 ** depth * (p + 1) ** 2 * 4)
    s.passes(q)
    assert all(np.array_equal(a, b) for a, b in zip(levels(), want))
    s.close()


@pytest.mark.parametrize("row", [4, 36, 1352, 4608])
@pytest.mark.parametrize("n", [0, 1, 5, 63])
def test_clear_rows(wb, row, n):
    rng = np.random.default_rng(row + n)
    rows, planes = 64, 3
    a = rng.integers(1, 255, (planes, rows, row), dtype=np.uint8)
    lst = np.sort(rng.permutation(rows)[:n]).astype(np.uint32)
    d, dl = wb.DeviceBuffer.from_array(a), wb.DeviceBuffer.from_array(
        lst if n else np.zeros(1, np.uint32))
    f = wb.lib().wbfmm_hip_clear_rows
    vp, sz, u = ctypes.c_void_p, ctypes.c_size_t, ctypes.c_uint
    assert f(vp(d.ptr), vp(dl.ptr), u(n), sz(rows), sz(row), u(planes)) == 0
    wb.sync()
    a[:, lst] = 0
    assert np.array_equal(d.download(np.zeros_like(a)), a)
