"""Performance cases of the FMM path: whole solves through the public entry
points, from the smallest call to the largest configuration of the
benchmark.

A case is one solve of a stated size: points uniform in a cube or on the
unit sphere with N(0,1) strengths (the distributions of the benchmark and
the tests), an octree depth, expansion orders and a precision.  `prepare`
makes what a program holds before the solve (points and strengths on the
device, or in host memory for the callers of the C drop-in, and the solver
with its operator tables), `run` is one solve: tree build, upward and
downward passes, field at the targets.

Orders come from the accuracies the serving engine is asked for: 1e-4,
1e-6 and 1e-8 give Laplace orders 9, 13 and 20 and, at low frequency,
Helmholtz orders 16, 23 and 30; the benchmark's own configurations use 11
and 12.
"""

import ctypes
import math

import numpy as np
import torch

import wbfmm_amd as W
import wbfmm_amd.serve as serve

CUTOFF = 1e-6      # pairs closer than this are left out, as in the near field
DEVICE = "cuda"

SERVE_STREAMS = 8  # streams of the serving engine, as the benchmark has them


def listed():
    return [
        # the C drop-in called with host arrays on a small problem, box
        # mirror on: what a user of the reference's drivers has; launches,
        # copies and host work count most
        dict(name="lap_host_1k", kind="laplace", shape="cube", n=1000, ntgt=0, depth=2, order=8,
             precision=64, dipoles=False, field=3, host=True),
        # an ordinary device-resident solve with separate targets, ragged
        # sizes, accuracy 1e-6
        dict(name="lap_f64_20k", kind="laplace", shape="cube", n=20011, ntgt=13337, depth=3,
             order=13, precision=64, dipoles=False, field=3, host=False),
        # the benchmark's headline configuration
        dict(name="lap_f64_1m", kind="laplace", shape="cube", n=1000000, ntgt=0, depth=7, order=12,
             precision=64, dipoles=False, field=3, host=False),
        # accuracy 1e-8 with FP64 at the engine's depth for this size
        dict(name="lap_f64_200k_tight", kind="laplace", shape="cube", n=200003, ntgt=0, depth=5,
             order=20, precision=64, dipoles=False, field=3, host=False),
        # single-precision expansions at accuracy 1e-4
        dict(name="lap_f32_300k", kind="laplace", shape="cube", n=300000, ntgt=0, depth=5, order=9,
             precision=32, dipoles=False, field=3, host=False),
        # surface sources with normal dipoles (boundary-element use),
        # potential only, separate targets
        dict(name="lap_dipole_sphere_60k", kind="laplace", shape="sphere", n=60000, ntgt=31013,
             depth=5, order=10, precision=64, dipoles=True, field=1, host=False),
        # vector sources: the curl and its gradient (vortex methods)
        dict(name="lap_curl_30k", kind="curl", shape="cube", n=30000, ntgt=0, depth=4, order=10,
             precision=64, dipoles=False, field=6, host=False),
        # the benchmark's plain Helmholtz cube
        dict(name="hel_f64_cube_10k", kind="helmholtz", shape="cube", n=10000, ntgt=10000, depth=4,
             order=11, tol=0.0, k=1.0, precision=64, dipoles=False, field=3, host=False),
        # the benchmark's sphere scattering configuration, mixed precision
        dict(name="hel_mixed_sphere_1m", kind="helmholtz", shape="sphere", n=1000000, ntgt=0,
             depth=7, order=0, tol=1e-6, k=16.0, precision=32, dipoles=True, field=3, host=False),
        # the same kind of problem at a tenth of the size, all in FP64
        dict(name="hel_f64_sphere_100k", kind="helmholtz", shape="sphere", n=100003, ntgt=0,
             depth=5, order=0, tol=1e-6, k=16.0, precision=64, dipoles=True, field=3, host=False),
        # accuracy 1e-8: orders of 30 and above
        dict(name="hel_f64_cube_30k_tight", kind="helmholtz", shape="cube", n=30000, ntgt=0,
             depth=3, order=0, tol=1e-8, k=8.0, precision=64, dipoles=False, field=3, host=False),
        # a batch of uneven Laplace and Helmholtz problems through the
        # serving engine
        dict(name="serve_mix_16", kind="serve", count=16, lo=3.0, hi=4.7, tol=1e-6),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: the kinds above over their sizes, depths (leaves of a
    fraction of a point to some tens of points), orders and options."""
    kind = rng.choice(["laplace", "laplace", "laplace", "curl", "helmholtz", "helmholtz", "serve"])
    if kind == "serve":
        return dict(kind="serve", count=rng.randint(6, 16), lo=3.0,
                    hi=round(rng.uniform(3.8, 4.7), 2), tol=rng.choice([1e-4, 1e-6]))
    shape = rng.choice(["cube", "sphere"])
    if kind == "curl":
        n = _log(rng, 1000, 60000)
        return dict(kind=kind, shape="cube", n=n, ntgt=0, depth=_depth(rng, n, "cube", 5),
                    order=rng.randint(4, 13), precision=64, dipoles=False, field=rng.choice([4, 6]),
                    host=False)
    if kind == "laplace":
        n = _log(rng, 1000, 300000)
        precision = rng.choice([64, 64, 32])
        host = precision == 64 and n < 30000 and rng.random() < 0.3
        return dict(kind=kind, shape=shape, n=n,
                    ntgt=0 if rng.random() < 0.5 else _log(rng, 500, n + 500),
                    depth=_depth(rng, n, shape, 6),
                    order=rng.randint(4, 20) if precision == 64 else rng.randint(4, 15),
                    precision=precision, dipoles=rng.random() < 0.25, field=rng.choice([1, 3, 3]),
                    host=host)
    tol = rng.choice([1e-4, 1e-6, 1e-6, 1e-8])
    n = _log(rng, 1000, 150000 if tol > 1e-8 else 20000)
    return dict(kind=kind, shape=shape, n=n, ntgt=0 if rng.random() < 0.5 else _log(rng, 500, n + 500),
                depth=_depth(rng, n, shape, 5 if tol > 1e-8 else 3), order=0, tol=tol,
                k=round(rng.uniform(1.0, 16.0), 2),
                precision=rng.choice([64, 32]) if tol >= 1e-6 else 64,
                dipoles=shape == "sphere" and rng.random() < 0.5, field=rng.choice([1, 3, 3]),
                host=False)


def _depth(rng, n, shape, most):
    per = math.exp(rng.uniform(math.log(2.0), math.log(40.0)))
    branch = 8.0 if shape == "cube" else 4.1
    return max(2, min(most, int(round(math.log(max(n / per, 1.0)) / math.log(branch)))))


# ---------------------------------------------------------------- inputs

def _points(gen, n, shape, width=2.0):
    if shape == "sphere":
        x = torch.randn((n, 3), generator=gen, device=DEVICE, dtype=torch.float64)
        return x / x.norm(dim=1, keepdim=True)
    return width * (torch.rand((n, 3), generator=gen, device=DEVICE, dtype=torch.float64) - 0.5)


def _inputs(case, seed):
    """points, targets (None: the points), strengths, dipole strengths and
    normals of a case"""
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(int(seed))
    n = case["n"]
    cols = {"helmholtz": 2, "curl": 3}.get(case["kind"], 1)
    xs = _points(gen, n, case["shape"])
    q = torch.randn((n, cols), generator=gen, device=DEVICE, dtype=torch.float64)
    d = normals = None
    if case["dipoles"]:
        # half monopoles, half dipoles along unit normals
        d = torch.randn((n, cols), generator=gen, device=DEVICE, dtype=torch.float64)
        q[1::2] = 0.0
        d[0::2] = 0.0
        normals = xs.clone() if case["shape"] == "sphere" else _points(gen, n, "sphere")
    xt = _points(gen, case["ntgt"], "cube") if case["ntgt"] else None
    if xt is not None and case["shape"] == "sphere":
        xt *= 0.9      # a cube of field points that reaches through the surface
    return xs, xt, q, d, normals


def _domain(xs, xt):
    """min corner less 0.01 and the widest extent plus 0.02, as the drivers
    fit it"""
    lo, hi = xs.amin(0), xs.amax(0)
    if xt is not None:
        lo, hi = torch.minimum(lo, xt.amin(0)), torch.maximum(hi, xt.amax(0))
    lo, hi = lo.cpu().numpy(), hi.cpu().numpy()
    return lo - 0.01, float((hi - lo).max()) + 0.02


def _width(case):
    if case["kind"] == "curl":
        return 12 if case["field"] & 2 else 3
    c = 2 if case["kind"] == "helmholtz" else 1
    return c * ((1 if case["field"] & 1 else 0) + (3 if case["field"] & 2 else 0))


def _parts(f, kind, field):
    """the columns of a field array: the potential and its gradient, or the
    curl and its gradient"""
    first = 3 if kind == "curl" else (2 if kind == "helmholtz" else 1) if field & 1 else 0
    out = {}
    if first:
        out["curl" if kind == "curl" else "potential"] = f[:, :first]
    if field & 2:
        out["gradient"] = f[:, first:]
    return out


def _orders(case, D):
    if case["order"]:
        return [case["order"]] * 17
    t = W.WbfmmTree()
    t.D = D
    o = [W.lib().wbfmm_truncation_number(ctypes.byref(t), case["k"], max(l, 2), case["tol"])
         for l in range(case["depth"] + 1)]
    return o + [o[-1]] * (17 - len(o))


class _Solve:
    """A solver with its inputs and its output array."""

    def __init__(self, case, seed):
        self.case = case
        xs, xt, q, d, normals = _inputs(case, seed)
        x0, D = _domain(xs, xt)
        orders = _orders(case, D)
        width = _width(case)
        self.ntgt = case["n"] if xt is None else case["ntgt"]
        self.f = torch.zeros((self.ntgt, width), device=DEVICE, dtype=torch.float64)
        if case["host"]:
            get = lambda a: None if a is None else np.ascontiguousarray(a.cpu().numpy())
            xs, xt, q, d, normals = (get(a) for a in (xs, xt, q, d, normals))
            self.f = np.zeros((self.ntgt, width))
        self.xs, self.xt, self.q, self.d, self.normals = xs, xs if xt is None else xt, q, d, normals
        torch.cuda.synchronize()   # the library works on a stream of its own
        if case["kind"] == "helmholtz":
            self.solver = W.HelmholtzSolver(self.xs, x0, D, case["depth"], orders, orders, case["k"],
                                            normals=normals, targets=self.xt,
                                            precision=case["precision"])
        else:
            curl = case["kind"] == "curl"
            self.solver = W.LaplaceSolver(self.xs, x0, D, case["depth"], orders, orders,
                                          targets=None if curl else self.xt, normals=normals,
                                          precision=case["precision"], nq=3 if curl else 1,
                                          host_mirror=case["host"])

    def solve(self):
        c, s, width = self.case, self.solver, _width(self.case)
        if c["host"]:
            self.f[:] = 0.0
        else:
            # the field is accumulated: cleared on the library's stream
            W.lib().wbfmm_hip_memset(W.ptr(self.f), 0, self.f.numel() * 8)
        if c["kind"] == "laplace":
            s.solve(self.q, self.f, field=c["field"], fstr=width, d=self.d)
        elif c["kind"] == "curl":
            s.build_tree()
            s.passes(self.q, sstr=3)
            s.field_points(self.xt, self.q, self.f, field=c["field"], fstr=width, sstr=3)
        else:
            s.build_tree()
            s.passes(self.q, d=self.d)
            s.field(self.xt, self.q, self.f, field=c["field"], fstr=width, d=self.d)
        return _parts(self.f, c["kind"], c["field"])

    def __del__(self):
        if getattr(self, "solver", None) is not None:
            torch.cuda.synchronize()
            self.solver.close()


_server = None


def _engine():
    """the process's serving engine, as a server keeps one"""
    global _server
    if _server is None:
        _server = serve.Server(SERVE_STREAMS)
    return _server


def _mix(case):
    """sizes, kernels, shapes and wavenumbers of a served batch: sizes
    log-uniform, kernels alternating, cube or sphere"""
    out = []
    for i in range(case["count"]):
        u = (i + 0.5) / case["count"]
        out.append(dict(kind="helmholtz" if i % 2 else "laplace", shape="sphere" if i % 4 > 1 else "cube",
                        n=int(10.0 ** (case["lo"] + (case["hi"] - case["lo"]) * u)) + i,
                        k=1.0 + 19.0 * ((7 * i) % case["count"]) / case["count"]))
    return out


class _Batch:
    """A batch of problems for the serving engine."""

    def __init__(self, case, seed):
        self.case = case
        gen = torch.Generator(device=DEVICE)
        gen.manual_seed(int(seed))
        self.problems = []
        for p in _mix(case):
            hel = p["kind"] == "helmholtz"
            p["xs"] = _points(gen, p["n"], p["shape"])
            p["q"] = torch.randn((p["n"], 2 if hel else 1), generator=gen, device=DEVICE,
                                 dtype=torch.float64)
            p["f"] = torch.zeros((p["n"], 8 if hel else 4), device=DEVICE, dtype=torch.float64)
            self.problems.append(p)
        torch.cuda.synchronize()
        _engine()

    def solve(self):
        srv = _engine()
        for p in self.problems:
            W.lib().wbfmm_hip_memset(W.ptr(p["f"]), 0, p["f"].numel() * 8)
        W.sync()     # the engine adds into f on streams of its own
        tickets = []
        for p in self.problems:
            hel = p["kind"] == "helmholtz"
            tickets.append(srv.submit(serve.make_request(
                serve.WBFMM_PROBLEM_HELMHOLTZ if hel else serve.WBFMM_PROBLEM_LAPLACE, p["xs"],
                q=p["q"], f=p["f"], k=p["k"] if hel else 0.0, tol=self.case["tol"], field=3,
                precision=0)))
        for t in tickets:
            if srv.wait(t).status:
                raise RuntimeError("a served problem failed")
        return [_parts(p["f"], p["kind"], 3) for p in self.problems]


def prepare(case, seed):
    return (_Batch if case["kind"] == "serve" else _Solve)(case, seed)


def run(state):
    return state.solve()


# ------------------------------------------------------------- reference

def _laplace_direct(xs, xt, q, d, normals, field):
    """potential and gradient of sum q/(4 pi r) + d n.(x-y)/(4 pi r^3)"""
    cols = []
    for t in _chunks(xt, len(xs)):
        r = [t[:, None, a] - xs[None, :, a] for a in range(3)]
        r2 = r[0] * r[0] + r[1] * r[1] + r[2] * r[2]
        ir = torch.where(r2 > CUTOFF * CUTOFF, r2.rsqrt(), torch.zeros_like(r2))
        ir3 = ir * ir * ir
        pot = ir @ q
        grad = [-((r[a] * ir3) @ q) for a in range(3)]
        if d is not None:
            nr = r[0] * normals[:, 0] + r[1] * normals[:, 1] + r[2] * normals[:, 2]
            pot = pot + (nr * ir3) @ d
            if field & 2:
                m = nr * (3.0 * ir3 * ir * ir)
                grad = [grad[a] + ir3 @ (d * normals[:, a]) - (m * r[a]) @ d for a in range(3)]
        cols.append(torch.stack(([pot] if field & 1 else []) + (grad if field & 2 else []), 1))
    return torch.cat(cols) / (4.0 * math.pi)


def _curl_direct(xs, xt, q, field):
    """u = curl of the vector potential, and d_j u_i at 3 + 3 j + i"""
    cols = []
    for t in _chunks(xt, len(xs)):
        r = [t[:, None, a] - xs[None, :, a] for a in range(3)]
        r2 = r[0] * r[0] + r[1] * r[1] + r[2] * r[2]
        ir = torch.where(r2 > CUTOFF * CUTOFF, r2.rsqrt(), torch.zeros_like(r2))
        ir3 = ir * ir * ir
        ir5 = ir3 * ir * ir
        J = [[-((r[a] * ir3) @ q[:, l]) for a in range(3)] for l in range(3)]
        out = [J[2][1] - J[1][2], J[0][2] - J[2][0], J[1][0] - J[0][1]]
        if field & 2:
            H = [[None] * 3 for _ in range(3)]
            for a in range(3):
                for b in range(a, 3):
                    h = 3.0 * r[a] * r[b] * ir5
                    if a == b:
                        h = h - ir3
                    h = h @ q
                    H[a][b] = H[b][a] = h
            for j in range(3):
                out += [H[j][1][:, 2] - H[j][2][:, 1], H[j][2][:, 0] - H[j][0][:, 2],
                        H[j][0][:, 1] - H[j][1][:, 0]]
        cols.append(torch.stack(out, 1))
    return torch.cat(cols) / (4.0 * math.pi)


def _helmholtz_direct(xs, xt, q, d, normals, k, field):
    """potential and gradient of q G + d n.grad G, G = exp(ikr)/(4 pi i k r);
    the sums over real factors, real and imaginary parts apart"""
    cols = []
    z = q[:, 0] + 1j * q[:, 1]
    zd = None if d is None else d[:, 0] + 1j * d[:, 1]

    def mul(a, b, v):      # (a + i b) @ v
        v2 = torch.view_as_real(v).contiguous()
        x, y = a @ v2, b @ v2
        return torch.complex(x[:, 0] - y[:, 1], x[:, 1] + y[:, 0])

    for t in _chunks(xt, 2 * len(xs)):
        r = [t[:, None, a] - xs[None, :, a] for a in range(3)]
        rr = (r[0] * r[0] + r[1] * r[1] + r[2] * r[2]).sqrt()
        near = rr <= CUTOFF
        ir = torch.where(near, torch.zeros_like(rr), 1.0 / rr)
        s = ir / (4.0 * math.pi * k)
        g = (torch.sin(k * rr) * s, -torch.cos(k * rr) * s)      # G
        # G' = G (ik - 1/r)
        g1 = (-g[0] * ir - k * g[1], -g[1] * ir + k * g[0])
        pot = mul(g[0], g[1], z)
        u = [c * ir for c in r]
        grad = [mul(g1[0] * c, g1[1] * c, z) for c in u] if field & 2 else []
        if zd is not None:
            nr = u[0] * normals[:, 0] + u[1] * normals[:, 1] + u[2] * normals[:, 2]
            pot = pot + mul(g1[0] * nr, g1[1] * nr, zd)
            if field & 2:
                # G'' = G' (ik - 1/r) + G / r^2
                g2 = (-g1[0] * ir - k * g1[1] + g[0] * ir * ir, -g1[1] * ir + k * g1[0] + g[1] * ir * ir)
                m = [(g2[p] - g1[p] * ir) * nr for p in range(2)]
                h = [g1[p] * ir for p in range(2)]
                grad = [grad[a] + mul(m[0] * u[a], m[1] * u[a], zd)
                        + mul(h[0], h[1], zd * normals[:, a]) for a in range(3)]
        cols.append(torch.stack(([pot] if field & 1 else []) + grad, 1))
    f = torch.view_as_real(torch.cat(cols))
    return f.reshape(len(f), -1)


def _chunks(xt, n):
    step = max(1, (1 << 25) // n)
    return (xt[i:i + step] for i in range(0, len(xt), step))


def exact(case, seed):
    """the FP64 direct sum over all sources; None where the pairs are too
    many"""
    if case["kind"] == "serve":
        b = _Batch(case, seed)
        return [_parts(_helmholtz_direct(p["xs"], p["xs"], p["q"], None, None, p["k"], 3)
                       if p["kind"] == "helmholtz"
                       else _laplace_direct(p["xs"], p["xs"], p["q"][:, 0], None, None, 3),
                       p["kind"], 3)
                for p in b.problems]
    nt = case["ntgt"] or case["n"]
    if case["n"] * nt > (2.2e10 if case["kind"] == "helmholtz" else 9.1e10):
        return None
    xs, xt, q, d, normals = _inputs(case, seed)
    xt = xs if xt is None else xt
    if case["kind"] == "helmholtz":
        f = _helmholtz_direct(xs, xt, q, d, normals, case["k"], case["field"])
    elif case["kind"] == "curl":
        f = _curl_direct(xs, xt, q, case["field"])
    else:
        f = _laplace_direct(xs, xt, q[:, 0], None if d is None else d[:, 0], normals, case["field"])
    return _parts(f.cpu().numpy() if case["host"] else f, case["kind"], case["field"])


def tolerance(case):
    # FP64: another order of the translations' sums differs by 1e-16 (2-norm)
    # and 1e-15 (largest); a few hundred times that for another order within
    # the operators.  FP32 expansions: two FP32 kernels differ by 8e-8 and
    # either from FP64 by 3.3e-7 (potential), four times that here
    if case["kind"] == "serve" or case["precision"] == 32:
        return {"rel": 1.5e-6, "max": 1e-4}
    return {"rel": 1e-13, "max": 1e-10}


# ------------------------------------------------------------------ work

def _occupied(n, level, shape):
    """expected boxes of a level that hold one of n points, and boxes"""
    boxes = 8.0 ** level if shape == "cube" else 4.1 * 4.0 ** level
    return boxes * -math.expm1(-n / boxes), boxes


def _pairs(case, level):
    """expected (occupied target, occupied source) pairs of list 4"""
    nb = 2 ** level
    src, boxes = _occupied(case["n"], level, case["shape"])
    ntgt = max(case["n"], case["ntgt"]) if case["shape"] == "cube" else case["n"]
    tgt, _ = _occupied(ntgt, level, case["shape"])
    if case["shape"] == "sphere":
        return tgt * min(43.0, 0.5 * boxes) * src / boxes
    far = sum(min(nb - 1, i - i % 2 + 3) - max(0, i - i % 2 - 2) + 1 for i in range(nb)) ** 3
    near = sum(min(nb - 1, i + 1) - max(0, i - 1) + 1 for i in range(nb)) ** 3
    return (far - near) * (src / boxes) * (tgt / boxes)


def _flops(case, orders):
    """the translations of list 4 and between levels (two rotations and a
    coaxial shift with the blocks split by symmetry), the leaf expansions,
    the local fields and the near field"""
    hel = case["kind"] == "helmholtz"
    nq = 3 if case["kind"] == "curl" else 1
    nt = case["ntgt"] or case["n"]
    total = 0.0
    for level in range(2, case["depth"] + 1):
        N = orders[level]
        s = sum(j * j for j in range(1, N + 2)) + sum(j * j for j in range(1, N + 1))
        per = (16.0 if hel else 6.0) * s
        total += nq * _pairs(case, level) * per
        if level > 2:
            total += 2.0 * nq * _occupied(case["n"], level, case["shape"])[0] * per
    C = (orders[case["depth"]] + 1) ** 2
    total += nq * (case["n"] * C * (16.0 if hel else 6.0) + nt * C * (32.0 if hel else 16.0))
    leaves = 8.0 ** case["depth"] if case["shape"] == "cube" else 4.1 * 4.0 ** case["depth"]
    near = nt * case["n"] / leaves * (27.0 if case["shape"] == "cube" else 10.0)
    return total + nq * near * (60.0 if hel else 20.0)


def work(case):
    if case["kind"] == "serve":
        parts = []
        for p in _mix(case):
            hel = p["kind"] == "helmholtz"
            depth = max(2, int(round(math.log(p["n"] / (32.0 if hel else 16.0)) / math.log(8.0))))
            order = {1e-4: (9, 16), 1e-6: (13, 23), 1e-8: (20, 30)}[case["tol"]][1 if hel else 0]
            parts.append(work(dict(kind=p["kind"], shape=p["shape"], n=p["n"], ntgt=0, depth=depth,
                                   order=order, dipoles=False, field=3, k=p["k"])))
        return {key: sum(w[key] for w in parts) for key in ("bytes", "flops")}
    n, nt = case["n"], case["ntgt"] or case["n"]
    cols = {"helmholtz": 2, "curl": 3}.get(case["kind"], 1)
    read = n * 8.0 * (3 + cols + (3 + cols if case["dipoles"] else 0))
    read += 24.0 * case["ntgt"]
    return {"bytes": read + 8.0 * nt * _width(case), "flops": _flops(case, _orders(case, 2.02))}
