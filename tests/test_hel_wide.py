"""Helmholtz translations with run-time orders (hel_wide.hip): orders 28..40
and levels of two different orders.

CPU: the plan's slots, tiles and maps, and the tables applied with numpy as
the kernel applies them, against the oracle's rotate / coaxial shift /
rotate back.  GPU: whole solves against the oracle FMM, in each of the
kernel's ranges of orders (..24, ..31, ..40) and with unequal orders.
"""

import ctypes
import math
import os
import subprocess
import sys

import numpy as np
import pytest

from conftest import fit_box

MAXT, MAXU = 80, 861
_i, _d = ctypes.c_int, ctypes.c_double


class Plan(ctypes.Structure):
    """wbfmm_hel_wide_plan_t"""
    _fields_ = [("N", _i), ("NU", _i), ("KT", _i), ("NTH", _i), ("NR", _i), ("nt", _i * 2),
                ("wbeg", (_i * 17) * 2), ("tile", ((_i * 4) * MAXT) * 2),
                ("map1", (_i * (16 * MAXT)) * 2), ("map2", (_i * (16 * MAXT)) * 2),
                ("map3", (_i * (16 * MAXT)) * 2), ("s1", (_i * MAXU) * 2), ("th", _i * 343),
                ("rix", _i * 343), ("chi", _d * 343), ("rr", _d * 32)]


def make_plan(wb, N):
    P = Plan()
    assert wb.lib().wbfmm_hip_hel_wide_plan(N, ctypes.byref(P)) == 0
    return P


@pytest.mark.parametrize("N", range(2, 41))
def test_plan_slots_and_tiles(wb, N):
    P = make_plan(wb, N)
    NU = (N + 1) * (N + 2) // 2
    assert P.NU == NU and P.NTH == 49 and P.NR == 15
    # row tiles per part that the kernel's ranges of orders hold
    most = 32 if N <= 24 else 44 if N <= 31 else 72
    steps = []
    for pt in range(2):
        rows = NU if pt == 0 else NU - (N + 1)
        nt = P.nt[pt]
        assert nt <= most
        assert P.wbeg[pt][0] == 0 and P.wbeg[pt][16] == nt
        for w in range(16):
            assert 0 <= P.wbeg[pt][w + 1] - P.wbeg[pt][w] <= -(-most // 16)
        for t in range(nt):
            kb, nk, ko = P.tile[pt][t][0], P.tile[pt][t][1], P.tile[pt][t][2]
            # the kernel's buffer has three rows past the blocks, zeros or
            # rows of the other part, and 7, 8 or 11 k-steps at most
            assert 1 <= nk <= (7 if N <= 24 else 8 if N <= 31 else 11)
            assert 0 <= kb and kb + 4 * nk <= NU + 3
            steps.append((ko, nk))
        for m in (P.map1, P.map2):
            used = sorted(x for x in list(m[pt])[:16 * nt] if x >= 0)
            assert used == list(range(rows))
        units = sorted(x for x in list(P.map3[pt])[:16 * nt] if x >= 0)
        want = [n * (n + 1) // 2 + m for n in range(N + 1) for m in range(pt, n + 1)]
        assert units == sorted(want)
        s1 = [P.s1[pt][n * (n + 1) // 2 + m] for n in range(N + 1) for m in range(pt, n + 1)]
        assert sorted(s1) == list(range(rows))
    # the tables' k-steps are used once each, without a gap
    pos = 0
    for ko, nk in sorted(steps):
        assert ko == pos
        pos += nk
    assert pos == P.KT


def test_plan_refuses_orders_out_of_range(wb):
    P = Plan()
    for N in (-1, 0, 1, 41):
        assert wb.lib().wbfmm_hip_hel_wide_plan(N, ctypes.byref(P)) != 0


def apply_stage(P, pt, T, x):
    """rows of every tile of a part: T (KT, 64) in lane order on the slots x"""
    out = np.zeros(16 * P.nt[pt], complex)
    for t in range(P.nt[pt]):
        kb, nk, ko = P.tile[pt][t][0], P.tile[pt][t][1], P.tile[pt][t][2]
        for j in range(nk):
            A = T[ko + j].reshape(4, 16).T          # lane l: row l % 16, column l / 16
            out[16 * t:16 * t + 16] += A @ x[kb + 4 * j:kb + 4 * j + 4]
    return out


def emulate(P, T1, Ar, Ai, chi, M, N):
    L = np.zeros((N + 1) ** 2, complex)
    idx = lambda n, m: n * (n + 1) + m
    for pt in range(2):
        x = np.zeros(P.NU + 4, complex)
        for n in range(N + 1):
            for m in range(pt, n + 1):
                a = M[idx(n, m)] * np.exp(1j * m * chi)
                b = M[idx(n, -m)] * np.exp(-1j * m * chi)
                x[P.s1[pt][n * (n + 1) // 2 + m]] = a - b if pt else a + b

        def move(y, mp):
            z = np.zeros(P.NU + 4, complex)
            for r, s in enumerate(list(mp[pt])[:16 * P.nt[pt]]):
                if s >= 0:
                    z[s] = y[r]
            return z

        y = move(apply_stage(P, pt, T1, x), P.map1)
        z = apply_stage(P, pt, Ar, y)
        if Ai is not None:
            z = z + 1j * apply_stage(P, pt, Ai, y)
        u = move(apply_stage(P, pt, T1, move(z, P.map2)), P.map3)
        for n in range(N + 1):
            for nu in range(pt, n + 1):
                v = 0.5 * u[n * (n + 1) // 2 + nu]
                L[idx(n, nu)] += np.exp(-1j * nu * chi) * v
                if nu:
                    L[idx(n, -nu)] += np.exp(1j * nu * chi) * (-v if pt else v)
    return L


@pytest.mark.parametrize("N,Lt", [(3, 4), (17, 17), (28, 29)])
def test_tables_match_oracle(wb, oracle, N, Lt):
    lib = wb.lib()
    P = make_plan(wb, N)
    k, w = 2.3, 0.41
    ne = (Lt + 1) * (Lt + 2) * (Lt + 3) // 6
    rng = np.random.default_rng(300 + N)
    offs = [(2, 0, 0), (-3, 1, 2), (0, 0, -3), (3, -3, 3), (-2, -2, 0)]
    slots = [(a + 3) * 49 + (b + 3) * 7 + c + 3 for a, b, c in offs]
    th = np.array([oracle.shift_angles(*o)[0] for o in offs])
    A = np.zeros((len(offs), P.KT, 64))
    assert lib.wbfmm_hip_hel_wide_rot(ctypes.byref(P), len(offs), wb.ptr(th), wb.ptr(A)) == 0
    E = np.stack([oracle.hel_coaxial_table(1, Lt, k * w * P.rr[P.rix[s]])[:2 * ne] for s in slots])
    A2 = np.zeros((len(offs), 2, P.KT, 64))
    assert lib.wbfmm_hip_hel_wide_coax(ctypes.byref(P), Lt, len(offs), wb.ptr(E), wb.ptr(A2)) == 0
    M = np.zeros(2 * (N + 1) ** 2)
    for _ in range(3):
        oracle.hel_p2m(k, N, np.zeros(3), rng.uniform(-0.5, 0.5, 3) * w,
                       complex(*rng.normal(size=2)), M)
    for i, off in enumerate(offs):
        tho, ph, ch, r = oracle.shift_angles(*off)
        H = oracle.H_rotation(N, tho)
        Ef = oracle.hel_coaxial_table(1, Lt, k * w * r)
        Lref = oracle.hel_rotate(oracle.hel_coaxial(oracle.hel_rotate(M, N, H, ph, ch), N, N, Ef,
                                                    Lt, 1), N, H, ch, ph)
        Lref = Lref[0::2] + 1j * Lref[1::2]
        got = emulate(P, A[i], A2[i, 0], A2[i, 1], P.chi[slots[i]], M[0::2] + 1j * M[1::2], N)
        assert np.abs(got - Lref).max() < 1e-12 * np.abs(Lref).max(), off


def c2(z):
    return np.ascontiguousarray(np.stack([np.real(z), np.imag(z)], 1))


# orders of levels 2.. (source, receiver); the first level's are also those
# of levels 0 and 1
GPU_CASES = {
    "40": ([40, 40], [40, 40]),
    "31-30": ([31, 30], [31, 30]),
    "25-23": ([25, 23], [25, 23]),
    "unequal": ([9, 7], [6, 8]),
}


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(GPU_CASES))
def test_solve_matches_oracle(wb, oracle, name):
    # parity 1e-10 of each column's largest value, as for the other kernels;
    # 37 points leave chunks of 8 targets ragged at level 2 and most boxes
    # of level 3 empty
    os_, or_ = GPU_CASES[name]
    n = 37 if name == "40" else 700
    rng = np.random.default_rng(800)
    xs = rng.uniform(-1, 1, (n, 3))
    q = rng.normal(size=n) + 1j * rng.normal(size=n)
    k = 3.0
    x0, D = fit_box(xs)
    so = [os_[0], os_[0]] + os_ + [os_[-1]] * 13
    ro = [or_[0], or_[0]] + or_ + [or_[-1]] * 13
    print(f"orders {name}", flush=True)
    fs = []
    for rep in range(2):
        S = wb.HelmholtzSolver(xs, x0, D, 3, so, ro, k)
        S.build_tree()
        S.passes(c2(q))
        f = np.zeros((n, 8))
        S.field(xs, c2(q), f)
        wb.sync()
        S.close()
        fs.append(f)
    fo, _, _ = oracle.fmm(2, xs, xs, x0, D, 3, so, ro, q=c2(q), k=k, field=3, nthreads=8)
    for c in range(8):
        d = np.abs(fs[0][:, c] - fo[:, c]).max() / np.abs(fo[:, c]).max()
        assert d < 1e-10, (name, c, d)
    assert np.array_equal(fs[0], fs[1])


@pytest.mark.parametrize("Ns,Nr,level,nsrc,wide", [
    (28, 28, 5, 9, 1), (40, 28, 2, 9, 1), (27, 28, 7, 9, 1), (41, 41, 3, 9, 0), (1, 1, 3, 9, 0),
    (41, 20, 3, 9, 0),
    (27, 27, 3, 512, 0), (9, 9, 2, 64, 0),                       # equal: the per-order kernels
    (2, 1, 2, 9, 1), (9, 8, 3, 512, 1), (8, 9, 3, 9, 1),         # few targets
    (13, 12, 4, 3071, 0), (12, 13, 4, 9, 0), (14, 13, 4, 9, 1), (14, 13, 5, 9, 0),
    (15, 14, 5, 9, 1), (2, 15, 7, 9, 1),
    (11, 10, 4, 4096, 0), (12, 11, 4, 3072, 1), (11, 12, 10, 1 << 30, 1)])  # nearly full
def test_m2l_rule(wb, Ns, Nr, level, nsrc, wide):
    assert wb.lib().wbfmm_hip_hel_wide_m2l_serves(Ns, Nr, level, nsrc) == wide


@pytest.mark.gpu
@pytest.mark.parametrize("Ns,Nr,wide", [(5, 4, [1, 1, 0]), (4, 5, [1, 1, 0]), (14, 13, [1, 1, 1])])
def test_m2l_of_low_different_orders(wb, oracle, Ns, Nr, wide):
    """levels 2, 3 and 4 each on the kernel of the rule (the run-time-order one
    alone makes an occupancy bitmap), and the solve against the oracle FMM"""
    rng = np.random.default_rng(900)
    n, k, depth = 700, 2.0, 4
    xs, q = rng.uniform(-1, 1, (n, 3)), rng.normal(size=n) + 1j * rng.normal(size=n)
    x0, D = fit_box(xs)
    so, ro = [Ns] * 17, [Nr] * 17
    S = wb.HelmholtzSolver(xs, x0, D, depth, so, ro, k)
    S.build_tree()
    T = wb.Timing
    T.enable(True)
    T.reset()
    S.passes(c2(q))
    wb.sync()
    maps = T.query("m2l_occ_bits")[0]
    T.enable(False)
    assert maps == sum(wide)
    f = np.zeros((n, 8))
    S.field(xs, c2(q), f)
    S.close()
    fo, _, _ = oracle.fmm(2, xs, xs, x0, D, depth, so, ro, q=c2(q), k=k, field=3, nthreads=8)
    # parity 1e-10 of each column's largest value, as above
    assert (np.abs(f - fo).max(0) < 1e-10 * np.abs(fo).max(0)).all()


# counts the tables made, in front of the library's function
COUNT_C = r"""
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stdlib.h>
int made;
int wbfmm_hip_hel_wide_coax(const void *P, int L, int nr, const double *E, double *A2)
{
  int (*f)(const void *, int, int, const double *, double *);
  *(void **)&f = dlsym(dlopen(getenv("WBFMM_LIB"), RTLD_NOW | RTLD_NOLOAD), "wbfmm_hip_hel_wide_coax");
  made++;
  return f(P, L, nr, E, A2);
}
"""
COUNT_PY = r"""
import ctypes, os, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import numpy as np
import wbfmm_amd as wb
os.environ["WBFMM_LIB"] = wb.LIB_PATH
ctypes.CDLL(None).setenv(b"WBFMM_LIB", wb.LIB_PATH.encode(), 1)
rng = np.random.default_rng(1)
xs, q = rng.uniform(-1, 1, (300, 3)), rng.normal(size=(300, 2))
so, ro = [9, 9, 9, 8, 7] + [7] * 12, [6, 6, 6, 5, 4] + [4] * 12
S = wb.HelmholtzSolver(xs, np.full(3, -1.01), 2.02, 4, so, ro, 1.5)
made, fs = [], []
for rep in range(3):
    S.build_tree()
    S.passes(q)
    f = np.zeros((300, 8))
    S.field(xs, q, f)
    made.append(ctypes.c_int.in_dll(shim, "made").value)
    fs.append(f)
S.close()
assert np.array_equal(fs[0], fs[1]) and np.array_equal(fs[0], fs[2])
print("made", *made)
"""


@pytest.mark.gpu
def test_tables_are_made_once(tmp_path):
    """source and receiver orders differ, and between levels too: M2M and L2L
    ask for tables of different orders at each level, made by the first solve
    and kept for the next ones"""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    src, so = tmp_path / "count.c", tmp_path / "count.so"
    src.write_text(COUNT_C)
    r = subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(so), str(src), "-ldl"],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([sys.executable, "-u", "-c", COUNT_PY, str(so)], cwd=root,
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
    first, second, third = (int(a) for a in r.stdout.split()[-3:])
    assert first > 0 and second == third == first, r.stdout
