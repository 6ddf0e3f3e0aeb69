"""The field kernels give a target 1, 2, 4, 8 or 16 lanes, by the number of
targets.  The same targets evaluated in calls of different sizes (131072 and
more, 65536.., 32768.., 16384.., a few hundred: one case for each count, at
the edges) agree to rounding: the terms of a target's sum (at most 441
expansion terms and some hundred sources) are added in another order, each
order within 1e3 eps of the sum of the terms' magnitudes; 1e-12 of a column's
largest value.  The mixed-precision Helmholtz near field forms each source's
terms in FP32: some eight roundings of 6e-8, which the compiler may place
(fused or not) differently in each kernel; 5e-7.  The 16-lane kernels are compared with the oracle elsewhere."""

import numpy as np
import pytest

from conftest import fit_box

SIZES = [131073, 131072, 131071, 65536, 32769, 16384, 8193, 300, 1]
TOL = 1e-12


def points(seed, n):
    rng = np.random.default_rng(seed)
    xs = rng.uniform(0, 1, (n, 3))
    nrm = rng.normal(size=(n, 3))
    return rng, xs, nrm / np.linalg.norm(nrm, axis=1)[:, None]


def check(eval_at, xt, tol=TOL):
    """eval_at(targets) -> rows; the rows of every prefix agree"""
    ref = eval_at(np.ascontiguousarray(xt[:300]))
    scale = np.abs(ref).max(0)
    for m in SIZES:
        got = eval_at(np.ascontiguousarray(xt[:m]))
        assert np.all(np.isfinite(got))
        k = min(m, 300)
        d = (np.abs(got[:k] - ref[:k]).max(0) / scale).max()
        print(f"{m} targets: {d:.1e}", flush=True)
        assert d < tol, (m, d)


@pytest.mark.parametrize("n,nleaf,lanes", [
    # by the number of targets
    (1, 1, 16), (16383, 64, 16), (16384, 64, 8), (32767, 64, 8), (32768, 64, 4), (65536, 64, 2),
    (131072, 64, 1), (1 << 27, 1 << 30, 1),
    # four where the occupied leaves hold fewer than two each: 1e6 in a cube
    # and on a sphere at depth 7, 3e5 on a sphere at depths 6 and 7
    (1000000, 794000, 4), (1000000, 68200, 1), (300000, 17300, 1), (300000, 61700, 1),
    (300000, 178000, 4), (200000, 100000, 1), (200000, 100001, 4)])
def test_lanes_by_occupied_leaves(wb, n, nleaf, lanes):
    assert wb.lib().wbfmm_hip_lap_field_lanes(n, nleaf) == lanes


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [64, 32])
def test_empty_leaves_do_not_count(wb, precision):
    """140000 targets in few of the 262144 leaves of depth 6 take one lane
    each: the same bits as when each is asked for four times over, where the
    targets are more than twice all the leaves"""
    rng = np.random.default_rng(8)
    x = rng.normal(size=(140000, 3)) * 0.02 + 0.5
    xs, q = np.ascontiguousarray(x[::70]), rng.normal(size=2000)
    S = wb.LaplaceSolver(xs, np.zeros(3), 1.0, 6, [4] * 17, [4] * 17, precision=precision,
                         host_mirror=False)
    S.build_tree()
    S.passes(q)
    f, f4 = np.zeros((len(x), 4)), np.zeros((4 * len(x), 4))
    S.field_points(x, q, f)
    S.field_points(np.tile(x, (4, 1)), q, f4)
    S.close()
    assert np.abs(f).max() > 0 and np.array_equal(np.tile(f, (4, 1)), f4)


@pytest.mark.gpu
@pytest.mark.parametrize("precision,p,depth,dip", [(64, 1, 2, False), (64, 7, 3, True),
                                                   (64, 20, 2, False), (32, 9, 3, False)])
def test_laplace(wb, precision, p, depth, dip):
    rng, xs, nrm = points(11 + p, 3000)
    q, d = rng.normal(size=3000), rng.normal(size=3000)
    xt = rng.uniform(0, 1, (SIZES[0], 3))
    x0, D = fit_box(xs, xt)
    S = wb.LaplaceSolver(xs, x0, D, depth, [p] * 17, [p] * 17, normals=nrm, precision=precision,
                         host_mirror=False)
    dd = d if dip else None
    S.build_tree()
    S.passes(q, d=dd)

    def at(x):
        f = np.zeros((len(x), 4))
        S.field_points(x, q, f, field=3, fstr=4, d=dd)
        return f

    check(at, xt)
    S.close()


@pytest.mark.gpu
@pytest.mark.parametrize("field,width", [(6, 12), (4, 3), (3, 12)])
def test_vector_sources(wb, field, width):
    rng, xs, _ = points(31, 3000)
    q = np.ascontiguousarray(rng.normal(size=(3000, 3)))
    xt = rng.uniform(0, 1, (SIZES[0], 3))
    x0, D = fit_box(xs, xt)
    S = wb.LaplaceSolver(xs, x0, D, 3, [8] * 17, [8] * 17, nq=3, host_mirror=False)
    S.build_tree()
    S.passes(q, sstr=3)

    def at(x):
        f = np.zeros((len(x), width))
        S.field_points(x, q, f, field=field, fstr=width, sstr=3)
        return f

    check(at, xt)
    S.close()


@pytest.mark.gpu
@pytest.mark.parametrize("precision,p", [(64, 11), (32, 11), (64, 29)])
def test_helmholtz(wb, precision, p):
    # a third of the sources without a monopole, a third without a dipole
    rng, xs, nrm = points(51 + p, 3000)
    q, d = (np.ascontiguousarray(rng.normal(size=(3000, 2))) for _ in range(2))
    q[::3] = 0.0
    d[1::3] = 0.0
    xt = rng.uniform(0, 1, (SIZES[0], 3))
    x0, D = fit_box(xs, xt)
    S = wb.HelmholtzSolver(xs, x0, D, 3, [p] * 17, [p] * 17, 2.0, normals=nrm, precision=precision)
    S.build_tree()
    S.passes(q, d=d)

    def at(x):
        f = np.zeros((len(x), 8))
        S.field(x, q, f, field=3, fstr=8, d=d)
        return f

    check(at, xt, 5e-7 if precision == 32 else TOL)
    S.close()
