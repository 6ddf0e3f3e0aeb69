"""Helmholtz P2M at every number of table slots per thread (1..4: orders up
to 20, 29, 36 and 40) against the oracle: monopoles, dipoles, both; a box of
one point, of exactly one batch and of several; FP64 leaves, and FP32 leaves
scaled per degree."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def expansions(wb, oracle, N, bits, q, d, k, seed=0):
    """leaf expansions of a level-2 tree (download) and the oracle's"""
    rng = np.random.default_rng(seed)
    # boxes (0,0,0), (1,2,3) and (3,3,3) of 4^3: 1, 8 and 21 points, among
    # them one at a box centre and one on its polar axis
    cells = [(0, 0, 0)] + [(1, 2, 3)] * 8 + [(3, 3, 3)] * 21
    xs = (np.array(cells) + rng.uniform(0.02, 0.98, (30, 3))) / 4.0
    xs[3] = (np.array(cells[3]) + 0.5) / 4.0
    xs[12] = (np.array(cells[12]) + [0.5, 0.5, 0.9]) / 4.0
    nrm = rng.normal(size=(30, 3))
    nrm /= np.linalg.norm(nrm, axis=1)[:, None]
    qs = rng.normal(size=(30, 2)) if q else None
    ds = rng.normal(size=(30, 2)) if d else None
    orders = [0, 2, N]
    s = wb.HelmholtzSolver(xs, np.zeros(3), 1.0, 2, orders, orders, k, normals=nrm if d else None,
                           precision=bits)
    s.build_tree()
    lib = wb.lib()
    lib.wbfmm_tree_leaf_expansions(s.t, k, wb.ptr(qs), 2, wb.ptr(ds), 2, 1, None)
    got = s.coefficients(2, 0)
    s.close()
    box = np.array([sum(((c[a] >> b) & 1) << (3 * b + a) for b in range(2) for a in range(3))
                    for c in cells])
    want = np.zeros_like(got)
    for b in set(box):
        i = np.flatnonzero(box == b)
        x0 = (np.array(cells[i[0]]) + 0.5) / 4.0
        M = np.zeros(2 * (N + 1) ** 2)
        for j in i:
            if q:
                oracle.hel_p2m(k, N, x0, xs[j], qs[j, 0] + 1j * qs[j, 1], M)
            if d:
                oracle.hel_p2m_normal(k, N, x0, xs[j], nrm[j], ds[j, 0] + 1j * ds[j, 1], M)
        want[b] = M[0::2] + 1j * M[1::2]
    return got, want


@pytest.mark.parametrize("q,d", [(1, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("N", [2, 13, 20, 21, 29, 30, 36, 37, 40])
def test_p2m_orders(wb, oracle, N, q, d):
    got, want = expansions(wb, oracle, N, 64, q, d, 9.0, seed=N)
    # degree by degree, since j_n spans tens of decades: the recurrences and
    # the power lose about 2 N ulp, and the sums over 21 points as many again
    for n in range(N + 1):
        r = slice(n * n, (n + 1) ** 2)
        assert np.abs(got[:, r] - want[:, r]).max() <= 2e-13 * np.abs(want[:, r]).max(), n


@pytest.mark.parametrize("q,d", [(1, 0), (1, 1)])
@pytest.mark.parametrize("N", [12, 23, 27])
def test_p2m_scaled(wb, oracle, N, q, d):
    got, want = expansions(wb, oracle, N, 32, q, d, 2.0, seed=N)
    for n in range(N + 1):
        r = slice(n * n, (n + 1) ** 2)
        # rounded to FP32 once
        assert np.abs(got[:, r] - want[:, r]).max() <= 2 ** -23 * np.abs(want[:, r]).max(), n
