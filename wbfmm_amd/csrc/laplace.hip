// laplace.hip -- gfx950 kernels of the Laplace FMM path (FP64).
//
// Coefficients use the reference's real packing (n,0) at n^2, (n,m>0)
// re/im at n^2+2m-1, n^2+2m (src/wbfmm-private.h:76); level arrays are
// box-major on the device (coef_at, hip_common.h).  Every translation is
// the reference's rotate -> coaxial shift -> rotate back sequence
// (src/pass-laplace.c:35-105, src/shift-laplace.c:225-789); the rotations
// are applied as real (2n+1)x(2n+1) blocks built on the host from the
// Gumerov-Duraiswami H coefficients, and the coaxial shifts from the closed
// forms of src/laplace.c:542-725.
//
// Kernel shapes (first version, one wavefront per box):
//   P2M   one thread per occupied leaf box, column-wise Legendre recursion
//   M2M   one wave per parent, the 8 children staged through LDS
//   M2L   one wave per target box, list-4 sources streamed through LDS,
//         accumulators in registers (rows lane, lane+64, ...)
//   L2L   one wave per parent, its local expansion staged in LDS
//   L2P+P2P 1 to 16 lanes per target

#include <hip/hip_runtime.h>

#include <mutex>

#include "hip_common.h"

namespace wbfmm {

constexpr int kMaxN = WBFMM_HIP_MAX_ORDER;
constexpr int kRmax = ((kMaxN + 1) * (kMaxN + 1) + kWave - 1) / kWave;

// row r = n^2 + j of a block-diagonal rotation applied to x (LDS)
__device__ __forceinline__ double rot_row(const double *__restrict__ R,
                                          const double *x, int r) {
  int n = isqrt_deg(r), j = r - n * n, w = 2 * n + 1;
  const double *row = R + (size_t)n * (2 * n - 1) * (2 * n + 1) / 3 + j * w;
  const double *xb = x + n * n;
  double s = 0.0;
  for (int k = 0; k < w; k++) s = fma(row[k], xb[k], s);
  return s;
}

// coaxial tables: c[kind][(m*(L+1)+n)*(L+1)+nu]
__device__ __forceinline__ const double *coax_row(const double *cf, int L,
                                                  int m, int n) {
  return cf + ((size_t)m * (L + 1) + n) * (L + 1);
}

// The factors of the regular functions' recurrences and of the gradient per
// (j, k), 0 <= k <= j, and the ladder factors of the second derivatives:
// one table per process, built once on the device, read instead of several
// square roots and divisions per step.
struct LapCol {
  double al, be;      // P_j^k = Cth al P_{j-1}^k - be P_{j-2}^k (j > k)
  double f0, f1, f2;  // d/dz, and D+ from L_{j+1}^{k-1} and L_{j+1}^{k+1}
  double dg;          // P_k^k = dg Sth P_{k-1}^{k-1} (at j = k > 0)
  double rj;          // 1 / (2 j + 1)
  double pad;
};
constexpr int kLapTabN = WBFMM_HIP_MAX_ORDER + 3;
struct LapTab {
  LapCol c[(WBFMM_HIP_MAX_ORDER + 1) * (WBFMM_HIP_MAX_ORDER + 2) / 2];
  double la[kLapTabN][kLapTabN];          // lad_a(n, m)
  double lb[kLapTabN][2 * kLapTabN + 1];  // lad_s(mu) lad_b(n, mu), mu - kLapTabN
};

__device__ __forceinline__ double lad_kn(int n) { return (2.0 * n + 1) / (2.0 * n - 1); }
__device__ __forceinline__ double lad_a(int n, int m) {
  return n >= 1 && m <= n ? sqrt(lad_kn(n) * (double)(n - m) * (double)(n + m)) : 0.0;
}
__device__ __forceinline__ double lad_b(int n, int mu) {
  const double v = (double)(n - mu) * (double)(n - mu - 1);
  return (n >= 1 && v > 0.0) ? sqrt(lad_kn(n) * v) : 0.0;
}
__device__ __forceinline__ double lad_s(int mu) { return mu >= 0 ? -1.0 : 1.0; }

__global__ void k_lap_tab(LapTab *T) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < (WBFMM_HIP_MAX_ORDER + 1) * (WBFMM_HIP_MAX_ORDER + 2) / 2) {
    int j = 0;
    while ((j + 1) * (j + 2) / 2 <= t) j++;
    const int k = t - j * (j + 1) / 2, n1 = j + 1;
    LapCol c = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 1.0 / (2 * j + 1), 0.0};
    if (j > k) {
      const double h = sqrt((2.0 * j + 1) / (double)(j * j - k * k));
      c.al = sqrt(2.0 * j - 1) * h;
      c.be = j - 1 > k ? sqrt((double)((j - 1) * (j - 1) - k * k) / (2 * j - 3)) * h : 0.0;
    } else if (k > 0) {
      c.dg = sqrt((2.0 * k + 1) / (2.0 * k));
    }
    const double fc = sqrt((2.0 * n1 + 1) / (2.0 * n1 - 1));
    c.f0 = fc * sqrt((double)(n1 - k) * (n1 + k));
    c.f1 = k >= 1 ? fc * sqrt((double)(n1 - k + 1) * (n1 - k)) : 0.0;
    c.f2 = fc * sqrt((double)(n1 + k + 1) * (n1 + k));
    T->c[t] = c;
  }
  if (t < kLapTabN * kLapTabN) T->la[t / kLapTabN][t % kLapTabN] = lad_a(t / kLapTabN, t % kLapTabN);
  if (t < kLapTabN * (2 * kLapTabN + 1)) {
    const int n = t / (2 * kLapTabN + 1), mu = t % (2 * kLapTabN + 1) - kLapTabN;
    T->lb[n][mu + kLapTabN] = (mu < 0 ? -mu : mu) <= n ? lad_s(mu) * lad_b(n, mu) : 0.0;
  }
}

// ---------------------------------------------------------------------
// P2M (src/laplace.c:35-129, :315-423, :854-989)
// ---------------------------------------------------------------------
// T: coefficient type.  rs scales distances (1 for the reference's
// coefficients; 1/w for coefficients scaled by the box width, M_n / w^n,
// which the FP32 passes use): the recurrences run in FP64 either way.
template <typename T>
__global__ void k_lap_p2m(const uint32_t *boxes, unsigned nbox,
                          const uint32_t *start, const uint32_t *end,
                          const double *xyz, const double *q,
                          const double *nrm, const double *dip, int level,
                          double x0, double y0, double z0, double D, int N,
                          double rs, T *mps) {
  unsigned t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nbox) return;
  uint64_t b = boxes[t];
  uint32_t bi = compact3(b), bj = compact3(b >> 1), bk = compact3(b >> 2);
  double w = D / (double)(1u << level);
  double xc = x0 + w * (bi + 0.5), yc = y0 + w * (bj + 0.5),
         zc = z0 + w * (bk + 0.5);
  const int C = (N + 1) * (N + 1);
  const double s4pi = 1.0 / sqrt(4.0 * kPi);
  for (uint32_t s = start[b]; s < end[b]; s++) {
    double dx = xyz[4 * (size_t)s] - xc, dy = xyz[4 * (size_t)s + 1] - yc,
           dz = xyz[4 * (size_t)s + 2] - zc;
    double r = sqrt(dx * dx + dy * dy + dz * dz), rho = sqrt(dx * dx + dy * dy);
    double Cth = r > 0.0 ? dz / r : 1.0, Sth = r > 0.0 ? rho / r : 0.0;
    double cp = rho > 0.0 ? dx / rho : 1.0, sp = rho > 0.0 ? dy / rho : 0.0;
    // the dipole terms of M_{n+1} are built from R_n: one factor rs more
    double qs = q ? q[s] : 0.0, ds = dip ? dip[s] * rs : 0.0;
    const double rr = r * rs;
    double nx = 0, ny = 0, nz = 0;
    if (dip) {
      nx = nrm[4 * (size_t)s];
      ny = nrm[4 * (size_t)s + 1];
      nz = nrm[4 * (size_t)s + 2];
    }
    // nu+ = (nx - i ny)/2, nu- = (nx + i ny)/2 (dipole streaming form)
    double pmm = s4pi, rm = 1.0, cm = 1.0, sm = 0.0;
    for (int m = 0; m <= N; m++) {
      if (m > 0) {
        pmm *= sqrt((2.0 * m + 1) / (2.0 * m)) * Sth;
        rm *= rr;
        double tcm = cm * cp - sm * sp;
        sm = sm * cp + cm * sp;
        cm = tcm;
      }
      double p1 = 0.0, p0 = pmm, rn = rm;
      for (int n = m; n <= N; n++) {
        if (n > m) {
          double pn = (Cth * sqrt(2.0 * (n - 1) + 1) * p0 -
                       sqrt((double)((n - 1) * (n - 1) - m * m) / (2 * (n - 1) - 1)) * p1) *
                      sqrt((2.0 * (n - 1) + 3) / (double)(n * n - m * m));
          p1 = p0;
          p0 = pn;
          rn *= rr;
        }
        // R_n^m(y) = rn p0 e^{i m phi}
        double Rr = rn * p0 * cm, Ri = rn * p0 * sm;
        if (qs != 0.0) {
          double f = qs / (2 * n + 1);
          if (m == 0)
            mps[coef_at(b, n * n, C)] += f * Rr;
          else {
            mps[coef_at(b, n * n + 2 * m - 1, C)] += f * Rr;
            mps[coef_at(b, n * n + 2 * m, C)] -= f * Ri;
          }
        }
        if (ds != 0.0 && n < N) {
          // streaming form of M_{n+1} += d conj(nrm . grad R_{n+1})/(2n+3)
          int np = n + 1;
          double fc = sqrt((2.0 * np + 1) / (2.0 * np - 1)) * ds / (2 * np + 1);
          // (a) M_{n+1}^m += nz a conj(R_n^m)
          double a = fc * sqrt((double)(np - m) * (np + m));
          if (m == 0)
            mps[coef_at(b, np * np, C)] += nz * a * Rr;
          else {
            mps[coef_at(b, np * np + 2 * m - 1, C)] += nz * a * Rr;
            mps[coef_at(b, np * np + 2 * m, C)] -= nz * a * Ri;
          }
          // (b) M_{n+1}^{m-1}: -b1_{n+1}^{m-1} conj(nu+ R_n^m)
          if (m >= 1) {
            int mm = m - 1;
            double b1 = fc * sqrt((double)(np - mm) * (np - mm - 1));
            double ur = 0.5 * nx, ui = -0.5 * ny;  // nu+
            double vr = ur * Rr - ui * Ri, vi = ur * Ri + ui * Rr;
            if (mm == 0)
              mps[coef_at(b, np * np, C)] += -b1 * 2.0 * vr;
            else {
              mps[coef_at(b, np * np + 2 * mm - 1, C)] += -b1 * vr;
              mps[coef_at(b, np * np + 2 * mm, C)] -= -b1 * vi;
            }
          }
          // (c) M_{n+1}^{m+1}: b2_{n+1}^{m+1} conj(nu- R_n^m)
          {
            int mp = m + 1;
            double b2 = fc * sqrt((double)(np + mp) * (np + mp - 1));
            double ur = 0.5 * nx, ui = 0.5 * ny;  // nu-
            double vr = ur * Rr - ui * Ri, vi = ur * Ri + ui * Rr;
            mps[coef_at(b, np * np + 2 * mp - 1, C)] += b2 * vr;
            mps[coef_at(b, np * np + 2 * mp, C)] -= b2 * vi;
          }
        }
      }
    }
  }
}

// ---------------------------------------------------------------------
// Monopole P2M for leaves of a few points.  A group of L = N/2 + 1 lanes
// takes one box; lane j computes columns m = j and m = N - j of the regular
// solid harmonics (the middle column alone when N is even), so that every
// lane runs about N + 2 steps of the recurrence in n per point.  Each
// coefficient has one owner lane, which adds the box's points in source
// order in registers and then adds that sum to the box's expansion once.
// The arithmetic per point is that of k_lap_p2m (the square-root factors
// come from an LDS table that the block fills with the same expressions);
// what goes is k_lap_p2m's read-modify-write of every coefficient in
// global memory per point, a chain of dependent memory round trips.
// ---------------------------------------------------------------------
template <typename T, int NB>
__global__ __launch_bounds__(256) void k_lap_p2m_cols(
    const uint32_t *boxes, unsigned nbox, const uint32_t *start, const uint32_t *end,
    const double *xyz, const double *q, int level, double x0, double y0, double z0,
    double D, int N, double rs, T *mps) {
  constexpr int K = NB + 1;
  __shared__ double tA[K], tS[K], tB[K * K], tC[K * K];
  for (int i = threadIdx.x; i < K * K; i += blockDim.x) {
    const int k = i / K, m = i - (i / K) * K;
    if (m <= k) {
      // the factors of P_{k+1}^m from P_k^m and P_{k-1}^m
      tB[i] = sqrt((double)(k * k - m * m) / (2 * k - 1));
      tC[i] = sqrt((2.0 * k + 3) / (double)((k + 1) * (k + 1) - m * m));
    }
    if (i < K) {
      tA[i] = sqrt(2.0 * i + 1);
      tS[i] = i > 0 ? sqrt((2.0 * i + 1) / (2.0 * i)) : 0.0;
    }
  }
  __syncthreads();
  const int L = N / 2 + 1, BPW = 64 / L;
  const int lane = threadIdx.x & 63, g = lane / L, j = lane - g * L;
  const unsigned t = (blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * BPW + g;
  if (g >= BPW || t >= nbox) return;
  const int m1 = j, m2 = N - j;
  const bool pair = m2 > m1;
  const int sw = N - j + 1;               // first step of column m2
  const int last = pair ? N + 1 : N - j;  // last step of the lane
  const uint64_t b = boxes[t];
  const uint32_t bi = compact3(b), bj = compact3(b >> 1), bk = compact3(b >> 2);
  const double w = D / (double)(1u << level);
  const double xc = x0 + w * (bi + 0.5), yc = y0 + w * (bj + 0.5), zc = z0 + w * (bk + 0.5);
  const double s4pi = 1.0 / sqrt(4.0 * kPi);
  double ar[NB + 2], ai[NB + 2];
#pragma unroll
  for (int i = 0; i < NB + 2; i++) ar[i] = ai[i] = 0.0;
  for (uint32_t s = start[b]; s < end[b]; s++) {
    const double qs = q[s];
    if (qs == 0.0) continue;
    const double dx = xyz[4 * (size_t)s] - xc, dy = xyz[4 * (size_t)s + 1] - yc,
                 dz = xyz[4 * (size_t)s + 2] - zc;
    const double r = sqrt(dx * dx + dy * dy + dz * dz), rho = sqrt(dx * dx + dy * dy);
    const double Cth = r > 0.0 ? dz / r : 1.0, Sth = r > 0.0 ? rho / r : 0.0;
    const double cp = rho > 0.0 ? dx / rho : 1.0, sp = rho > 0.0 ? dy / rho : 0.0;
    const double rr = r * rs;
    // P_m^m, r^m and e^{i m phi} up to m2, kept at m1 on the way
    double pmm = s4pi, rm = 1.0, cm = 1.0, sm = 0.0;
    double pa = pmm, ra = rm, ca = cm, sa = sm;
#pragma unroll
    for (int i = 1; i <= NB; i++) {
      if (i <= m2) {
        pmm *= tS[i] * Sth;
        rm *= rr;
        const double tcm = cm * cp - sm * sp;
        sm = sm * cp + cm * sp;
        cm = tcm;
        if (i == m1) {
          pa = pmm;
          ra = rm;
          ca = cm;
          sa = sm;
        }
      }
    }
    double p1 = 0.0, p0 = pa, rn = ra, c = ca, sn = sa;
    int n = m1, m = m1;
#pragma unroll
    for (int st = 0; st < NB + 2; st++) {
      if (st > last) break;
      if (st > 0) {
        if (pair && st == sw) {
          m = m2;
          n = m2;
          p1 = 0.0;
          p0 = pmm;
          rn = rm;
          c = cm;
          sn = sm;
        } else {
          const int k = n;
          n++;
          const double pn = (Cth * tA[k] * p0 - tB[k * K + m] * p1) * tC[k * K + m];
          p1 = p0;
          p0 = pn;
          rn *= rr;
        }
      }
      const double Rr = rn * p0 * c, Ri = rn * p0 * sn;
      const double f = qs / (2 * n + 1);
      ar[st] += f * Rr;
      ai[st] += f * Ri;
    }
  }
  const int C = (N + 1) * (N + 1);
  T *out = mps + (size_t)b * C;
  int n = m1, m = m1;
#pragma unroll
  for (int st = 0; st < NB + 2; st++) {
    if (st > last) break;
    if (st > 0) {
      if (pair && st == sw) {
        m = m2;
        n = m2;
      } else {
        n++;
      }
    }
    if (m == 0) {
      out[n * n] += ar[st];
    } else {
      out[n * n + 2 * m - 1] += ar[st];
      out[n * n + 2 * m] -= ai[st];
    }
  }
}

// ---------------------------------------------------------------------
// The same expansions with one wavefront per box, for boxes that hold many
// points (clustered or small problems, where one thread per box leaves
// most of the chip idle and serialises hundreds of points).  The box's
// points are dealt to the wavefront's 64/GS groups of GS lanes, point
// start + i to group i mod (64/GS); lane m of a group computes column m of
// the regular solid harmonics (n = m..N) of its group's points and adds
// the monopole and dipole terms into the group's copy of the expansion in
// LDS.  Each of the three dipole terms is a statement of its own, in which
// every lane writes a distinct coefficient; a wavefront's LDS operations
// complete in program order.  The groups' copies are added in group order
// and the sum added to the box's expansion: no atomics, the same bits on
// every run.
//
// The factors of the recurrences and of the dipole terms come from the table
// (with square roots and divisions per step: 200003 points at order 20 0.82
// -> 0.41 ms, 3e5 at order 9, FP32, 0.32 -> 0.17, 6e4 with dipoles at order
// 10 0.21 -> 0.10).
// ---------------------------------------------------------------------
template <typename T, int GS>
__global__ __launch_bounds__(64) void k_lap_p2m_wave(
    const uint32_t *boxes, unsigned nbox, const uint32_t *start, const uint32_t *end,
    const double *xyz, const double *q, const double *nrm, const double *dip, int level,
    double x0, double y0, double z0, double D, int N, double rs, T *mps,
    const LapTab *__restrict__ tab) {
  extern __shared__ double pacc[];  // (64 / GS) copies of C coefficients
  constexpr int G = 64 / GS;
  const int lane = threadIdx.x, g = lane / GS, m = lane % GS;
  const int C = (N + 1) * (N + 1);
  const unsigned t = blockIdx.x;
  if (t >= nbox) return;
  for (int i = lane; i < G * C; i += 64) pacc[i] = 0.0;
  __syncthreads();
  const uint64_t b = boxes[t];
  const uint32_t bi = compact3(b), bj = compact3(b >> 1), bk = compact3(b >> 2);
  const double w = D / (double)(1u << level);
  const double xc = x0 + w * (bi + 0.5), yc = y0 + w * (bj + 0.5), zc = z0 + w * (bk + 0.5);
  const double s4pi = 1.0 / sqrt(4.0 * kPi);
  double *acc = pacc + g * C;
  auto put = [&](int n, int mm, double re, double im) {
    if (mm == 0)
      acc[n * n] += re;
    else {
      acc[n * n + 2 * mm - 1] += re;
      acc[n * n + 2 * mm] -= im;
    }
  };
  for (uint32_t s = start[b] + g; s < end[b]; s += G) {
    if (m > N) continue;
    const double dx = xyz[4 * (size_t)s] - xc, dy = xyz[4 * (size_t)s + 1] - yc,
                 dz = xyz[4 * (size_t)s + 2] - zc;
    const double r = sqrt(dx * dx + dy * dy + dz * dz), rho = sqrt(dx * dx + dy * dy);
    const double Cth = r > 0.0 ? dz / r : 1.0, Sth = r > 0.0 ? rho / r : 0.0;
    const double cp = rho > 0.0 ? dx / rho : 1.0, sp = rho > 0.0 ? dy / rho : 0.0;
    const double qs = q ? q[s] : 0.0, ds = dip ? dip[s] * rs : 0.0;
    const double rr = r * rs;
    double nx = 0, ny = 0, nz = 0;
    if (dip) {
      nx = nrm[4 * (size_t)s];
      ny = nrm[4 * (size_t)s + 1];
      nz = nrm[4 * (size_t)s + 2];
    }
    // P_m^m, r^m and e^{i m phi} of this lane's column
    double pmm = s4pi, rm = 1.0, cm = 1.0, sm = 0.0;
    for (int i = 1; i <= m; i++) {
      pmm *= tab->c[i * (i + 1) / 2 + i].dg * Sth;
      rm *= rr;
      const double tcm = cm * cp - sm * sp;
      sm = sm * cp + cm * sp;
      cm = tcm;
    }
    double p1 = 0.0, p0 = pmm, rn = rm;
    for (int n = m; n <= N; n++) {
      const LapCol tc = tab->c[n * (n + 1) / 2 + m];
      if (n > m) {
        const double pn = Cth * tc.al * p0 - tc.be * p1;
        p1 = p0;
        p0 = pn;
        rn *= rr;
      }
      const double Rr = rn * p0 * cm, Ri = rn * p0 * sm;
      if (qs != 0.0) {
        const double f = qs * tc.rj;
        put(n, m, f * Rr, f * Ri);
      }
      if (ds != 0.0 && n < N) {
        // streaming form of M_{n+1} += d conj(nrm . grad R_{n+1})/(2n+3),
        // as in k_lap_p2m: (a) column m, (b) column m - 1, (c) column m + 1
        const int np = n + 1;
        const double fc = ds / (2 * np + 1);
        const double a = fc * tc.f0;
        put(np, m, nz * a * Rr, nz * a * Ri);
        if (m >= 1) {
          const int mm = m - 1;
          const double b1 = fc * tc.f1;
          const double ur = 0.5 * nx, ui = -0.5 * ny;  // nu+
          const double vr = ur * Rr - ui * Ri, vi = ur * Ri + ui * Rr;
          if (mm == 0)
            acc[np * np] += -b1 * 2.0 * vr;
          else
            put(np, mm, -b1 * vr, -b1 * vi);
        }
        {
          const int mp = m + 1;
          const double b2 = fc * tc.f2;
          const double ur = 0.5 * nx, ui = 0.5 * ny;  // nu-
          const double vr = ur * Rr - ui * Ri, vi = ur * Ri + ui * Rr;
          put(np, mp, b2 * vr, b2 * vi);
        }
      }
    }
  }
  __syncthreads();
  for (int c = lane; c < C; c += 64) {
    double v = pacc[c];
#pragma unroll
    for (int h = 1; h < G; h++) v += pacc[h * C + c];
    mps[coef_at(b, c, C)] += (T)v;
  }
}

// ---------------------------------------------------------------------
// M2M (src/pass-laplace.c:433-486, src/shift-laplace.c:225-442)
// ---------------------------------------------------------------------
__global__ __launch_bounds__(64) void k_lap_m2m(
    const uint32_t *parents, unsigned npar, const uint32_t *cstart,
    const uint32_t *cend, double t, int Nc, int Np, const double *mps_c,
    double *mps_p, const double *rfwd, const double *rback, size_t nrot,
    const double *cf_ss, int L) {
  extern __shared__ double sh[];
  const int Cc = (Nc + 1) * (Nc + 1), Cp = (Np + 1) * (Np + 1);
  double *x = sh, *y = x + Cc, *z = y + Cc, *tp = z + Cp;
  const int lane = threadIdx.x;
  uint64_t p = parents[blockIdx.x];
  for (int k = lane; k <= Np; k += kWave) tp[k] = pow(-t, (double)k);
  double acc[kRmax];
#pragma unroll
  for (int q = 0; q < kRmax; q++) acc[q] = 0.0;
  for (int c = 0; c < 8; c++) {
    uint64_t cb = 8 * p + c;
    if (cend[cb] <= cstart[cb]) continue;
    __syncthreads();
    for (int r = lane; r < Cc; r += kWave) x[r] = mps_c[coef_at(cb, r, Cc)];
    __syncthreads();
    for (int r = lane; r < Cc; r += kWave)
      y[r] = rot_row(rfwd + c * nrot, x, r);
    __syncthreads();
    for (int r = lane; r < Cp; r += kWave) {
      int n = isqrt_deg(r), j = r - n * n, m = (j + 1) / 2;
      const double *cr = coax_row(cf_ss, L, m, n);
      double s = 0.0;
      int hi = n < Nc ? n : Nc;
      for (int nu = m; nu <= hi; nu++)
        s = fma(cr[nu] * tp[n - nu], y[nu * nu + j], s);
      z[r] = s;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kRmax; q++) {
      int r = lane + kWave * q;
      if (r < Cp) acc[q] += rot_row(rback + c * nrot, z, r);
    }
  }
#pragma unroll
  for (int q = 0; q < kRmax; q++) {
    int r = lane + kWave * q;
    if (r < Cp) mps_p[coef_at(p, r, Cp)] = acc[q];
  }
}

// ---------------------------------------------------------------------
// M2L (src/pass-laplace.c:35-105, :360-408)
// ---------------------------------------------------------------------
__global__ __launch_bounds__(64) void k_lap_m2l(
    const uint32_t *targets, unsigned ntgt, const uint32_t *sstart,
    const uint32_t *send, int level, double w, int Ns, int Nr,
    const double *mps, double *mpr, const double *rfwd, const double *rback,
    size_t nrot, const double *roff, const double *cf_sr, int L) {
  extern __shared__ double sh[];
  const int Cs = (Ns + 1) * (Ns + 1), Cr = (Nr + 1) * (Nr + 1);
  double *x = sh, *y = x + Cs, *z = y + Cs, *ipw = z + Cr;
  const int lane = threadIdx.x;
  uint64_t tb = targets[blockIdx.x];
  int ti = compact3(tb), tj = compact3(tb >> 1), tk = compact3(tb >> 2);
  int nbox = 1 << level;
  int i0 = ti - (ti & 1) - 2, j0 = tj - (tj & 1) - 2, k0 = tk - (tk & 1) - 2;
  double acc[kRmax];
#pragma unroll
  for (int q = 0; q < kRmax; q++) acc[q] = 0.0;
  for (int ii = i0; ii < i0 + 6; ii++) {
    if (ii < 0 || ii >= nbox) continue;
    for (int jj = j0; jj < j0 + 6; jj++) {
      if (jj < 0 || jj >= nbox) continue;
      for (int kk = k0; kk < k0 + 6; kk++) {
        if (kk < 0 || kk >= nbox) continue;
        int dx = ii - ti, dy = jj - tj, dz = kk - tk;
        if (dx >= -1 && dx <= 1 && dy >= -1 && dy <= 1 && dz >= -1 && dz <= 1)
          continue;
        uint64_t sb = spread3(ii) | (spread3(jj) << 1) | (spread3(kk) << 2);
        if (send[sb] <= sstart[sb]) continue;
        int o = (dx + 3) * 49 + (dy + 3) * 7 + dz + 3;
        double tt = roff[o] * w;
        __syncthreads();
        for (int r = lane; r < Cs; r += kWave) x[r] = mps[coef_at(sb, r, Cs)];
        for (int k = lane; k <= Ns + Nr + 1; k += kWave)
          ipw[k] = pow(tt, -(double)k);
        __syncthreads();
        for (int r = lane; r < Cs; r += kWave)
          y[r] = rot_row(rfwd + o * nrot, x, r);
        __syncthreads();
        for (int r = lane; r < Cr; r += kWave) {
          int n = isqrt_deg(r), j = r - n * n, m = (j + 1) / 2;
          const double *cr = coax_row(cf_sr, L, m, n);
          double s = 0.0;
          for (int nu = m; nu <= Ns; nu++)
            s = fma(cr[nu] * ipw[n + nu + 1], y[nu * nu + j], s);
          z[r] = s;
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < kRmax; q++) {
          int r = lane + kWave * q;
          if (r < Cr) acc[q] += rot_row(rback + o * nrot, z, r);
        }
      }
    }
  }
#pragma unroll
  for (int q = 0; q < kRmax; q++) {
    int r = lane + kWave * q;
    if (r < Cr) mpr[coef_at(tb, r, Cr)] += acc[q];
  }
}

// ---------------------------------------------------------------------
// L2L (src/pass-laplace.c:410-428, src/shift-laplace.c:562-789)
// ---------------------------------------------------------------------
__global__ __launch_bounds__(64) void k_lap_l2l(
    const uint32_t *parents, unsigned npar, const uint32_t *cflag, double t,
    int Np, int Nc, const double *mpr_p, double *mpr_c, const double *rfwd,
    const double *rback, size_t nrot, const double *cf_rr, int L) {
  extern __shared__ double sh[];
  const int Cp = (Np + 1) * (Np + 1), Cc = (Nc + 1) * (Nc + 1);
  double *x = sh, *y = x + Cp, *z = y + Cp, *tp = z + Cc;
  const int lane = threadIdx.x;
  uint64_t p = parents[blockIdx.x];
  for (int r = lane; r < Cp; r += kWave) x[r] = mpr_p[coef_at(p, r, Cp)];
  for (int k = lane; k <= Np; k += kWave) tp[k] = pow(t, (double)k);
  for (int c = 0; c < 8; c++) {
    uint64_t cb = 8 * p + c;
    if (cflag && !cflag[cb]) continue;
    __syncthreads();
    for (int r = lane; r < Cp; r += kWave)
      y[r] = rot_row(rfwd + c * nrot, x, r);
    __syncthreads();
    for (int r = lane; r < Cc; r += kWave) {
      int n = isqrt_deg(r), j = r - n * n, m = (j + 1) / 2;
      const double *cr = coax_row(cf_rr, L, m, n);
      double s = 0.0;
      int lo = n > m ? n : m;
      for (int nu = lo; nu <= Np; nu++)
        s = fma(cr[nu] * tp[nu - n], y[nu * nu + j], s);
      z[r] = s;
    }
    __syncthreads();
    for (int r = lane; r < Cc; r += kWave)
      mpr_c[coef_at(cb, r, Cc)] += rot_row(rback + c * nrot, z, r);
  }
}

// ---------------------------------------------------------------------
// L2P + near field (src/local-laplace.c:333-630, :1091-1336)
// ---------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ void lcoef(const T *mpr, uint64_t b, int C,
                                      int n, int m, double &re, double &im) {
  if (m == 0) {
    re = mpr[coef_at(b, n * n, C)];
    im = 0.0;
  } else {
    re = mpr[coef_at(b, n * n + 2 * m - 1, C)];
    im = mpr[coef_at(b, n * n + 2 * m, C)];
  }
}

// lcoef without a branch on m (both reads issued; the imaginary part 0
// for m = 0)
template <typename T>
__device__ __forceinline__ void lcoef_nb(const T *mpr, uint64_t b, int C, int n, int m,
                                         double &re, double &im) {
  const int ir = m ? n * n + 2 * m - 1 : n * n, ii = m ? n * n + 2 * m : n * n;
  re = mpr[coef_at(b, ir, C)];
  const double v = mpr[coef_at(b, ii, C)];
  im = m ? v : 0.0;
}

// G lanes per target (G a power of two): the columns k of the local
// expansion dealt back and forth (lane g takes g, 2G-1-g, 2G+g, ..: near
// equal numbers of steps), the neighbours' sources as in NearSplit, and the
// lanes' sums added at the end.  One lane per target leaves most of the
// chip idle below a few hundred thousand targets: 13337 targets, order 13,
// 39 points a leaf, are 209 wavefronts, each a chain of 105 expansion steps
// and 1050 pairs (0.55 ms); see field_lanes for the figures.
// T: coefficient type; rs as in k_lap_p2m (1/w for coefficients scaled by
// the box width, L_n w^(n+1): the expansion then gives phi w and grad w^2)
template <typename T, int G>
__global__ __launch_bounds__(128) void k_lap_field(
    const double *__restrict__ xt, const uint32_t *__restrict__ tid, unsigned ntgt,
    const uint32_t *__restrict__ start, const uint32_t *__restrict__ end,
    const double *__restrict__ xyz, const double *__restrict__ q,
    const double *__restrict__ nrm, const double *__restrict__ dip, int level, double x0,
    double y0, double z0, double D, int N, double rs, const T *__restrict__ mpr, int field,
    double *__restrict__ f, int fstr, const LapTab *__restrict__ tab) {
  const unsigned id = blockIdx.x * blockDim.x + threadIdx.x, t = id / G;
  const int g = (int)(id % G);
  if (t >= ntgt) return;  // the same in a group's lanes
  double px = xt[4 * (size_t)t], py = xt[4 * (size_t)t + 1],
         pz = xt[4 * (size_t)t + 2];
  uint64_t code = point_code(px, py, pz, x0, y0, z0, D);
  uint64_t b = code >> (3 * (20 - level));
  int bi = compact3(b), bj = compact3(b >> 1), bk = compact3(b >> 2);
  double w = D / (double)(1u << level);
  double dx = px - (x0 + w * (bi + 0.5)), dy = py - (y0 + w * (bj + 0.5)),
         dz = pz - (z0 + w * (bk + 0.5));
  double r = sqrt(dx * dx + dy * dy + dz * dz), rho = sqrt(dx * dx + dy * dy);
  double Cth = r > 0.0 ? dz / r : 1.0, Sth = r > 0.0 ? rho / r : 0.0;
  double cp = rho > 0.0 ? dx / rho : 1.0, sp = rho > 0.0 ? dy / rho : 0.0;
  const int C = (N + 1) * (N + 1);
  const double s4pi = 1.0 / sqrt(4.0 * kPi);
  double phi = 0.0, gz = 0.0, gpr = 0.0, gpi = 0.0;  // gp = D+ phi
  const bool want_g = (field & 2) != 0;
  const double rr = r * rs;
  // regular solid harmonics R_j^k column by column
  double pmm = s4pi, rm = 1.0, cm = 1.0, sm = 0.0;
  int k0 = 0;
  for (int cb = 0; cb <= N; cb += G) {
    const int k = (cb / G) & 1 ? cb + G - 1 - g : cb + g;
    if (k > N) continue;
    for (; k0 < k; k0++) {
      const int kk = k0 + 1;
      pmm *= tab->c[kk * (kk + 1) / 2 + kk].dg * Sth;
      rm *= rr;
      double tcm = cm * cp - sm * sp;
      sm = sm * cp + cm * sp;
      cm = tcm;
    }
    double p1 = 0.0, p0 = pmm, rn = rm;
    double wk = (k == 0) ? 1.0 : 2.0;
    for (int j = k; j <= N; j++) {
      const LapCol tc = tab->c[j * (j + 1) / 2 + k];
      if (j > k) {
        double pn = Cth * tc.al * p0 - tc.be * p1;
        p1 = p0;
        p0 = pn;
        rn *= rr;
      }
      double Rr = rn * p0 * cm, Ri = rn * p0 * sm;
      double lr, li;
      lcoef_nb(mpr, b, C, j, k, lr, li);
      phi += wk * (lr * Rr - li * Ri);
      if (want_g && j < N) {
        int n1 = j + 1;
        // the three coefficients of degree j + 1 read without branches, so
        // that their loads issue together: L^k, L^{k-1} (weight 0 at k = 0,
        // read at order 0 there), L^{k+1} (k + 1 <= j + 1 always)
        double l0r, l0i, lmr, lmi, lpr, lpi;
        const int mm = k >= 1 ? k - 1 : 0, mp = k + 1;
        lcoef_nb(mpr, b, C, n1, k, l0r, l0i);
        lcoef_nb(mpr, b, C, n1, mm, lmr, lmi);
        lcoef_nb(mpr, b, C, n1, mp, lpr, lpi);
        // dz: a_{j+1}^k L_{j+1}^k R_j^k
        gz += wk * tc.f0 * (l0r * Rr - l0i * Ri);
        // D+: -b1_{j+1}^{k-1} L_{j+1}^{k-1} R_j^k
        gpr -= tc.f1 * (lmr * Rr - lmi * Ri);
        gpi -= tc.f1 * (lmr * Ri + lmi * Rr);
        // D+: b2_{j+1}^{k+1} conj(L_{j+1}^{k+1} R_j^k)
        gpr += tc.f2 * (lpr * Rr - lpi * Ri);
        gpi -= tc.f2 * (lpr * Ri + lpi * Rr);
      }
    }
  }
  phi *= rs;
  gz *= rs * rs;
  double gx = gpr * (rs * rs), gy = gpi * (rs * rs);
  // near field over the 27 neighbours, cutoff |x-y| <= 1e-6
  const double c4 = 0.25 / kPi, cut2 = 1e-12;
  near_sources<G>(g, bi, bj, bk, level, start, end, [&](uint32_t s) {
    double rx = px - xyz[4 * (size_t)s], ry = py - xyz[4 * (size_t)s + 1],
           rz = pz - xyz[4 * (size_t)s + 2];
    double r2 = rx * rx + ry * ry + rz * rz;
    if (r2 <= cut2) return;
    double ir = rsqrt(r2), ir3 = ir * ir * ir;
    if (q) {
      double qs = q[s] * c4;
      phi += qs * ir;
      gx -= qs * rx * ir3;
      gy -= qs * ry * ir3;
      gz -= qs * rz * ir3;
    }
    if (dip) {
      double nx = nrm[4 * (size_t)s], ny = nrm[4 * (size_t)s + 1],
             nz = nrm[4 * (size_t)s + 2];
      double nr = nx * rx + ny * ry + nz * rz, ds = dip[s] * c4;
      double ir5 = ir3 * ir * ir;
      phi += ds * nr * ir3;
      gx += ds * (nx * ir3 - 3.0 * nr * rx * ir5);
      gy += ds * (ny * ir3 - 3.0 * nr * ry * ir5);
      gz += ds * (nz * ir3 - 3.0 * nr * rz * ir5);
    }
  });
  phi = group_sum<G>(phi);
  gx = group_sum<G>(gx);
  gy = group_sum<G>(gy);
  gz = group_sum<G>(gz);
  if (g) return;
  double *out = f + (size_t)tid[t] * fstr;
  int o = 0;
  if (field & 1) out[o++] += phi;
  if (field & 2) {
    out[o++] += gx;
    out[o++] += gy;
    out[o++] += gz;
  }
}

// ---------------------------------------------------------------------
// Vector sources (nq components; src/local-laplace.c:333-630 per
// component, the curl :632-750 and :1013-1089 with near field :38-62, the
// curl and its gradient :752-1011 and :1229-1291 with near field :147-183).
// Component q's local expansions are plane q of the level array (plane
// stride pst).  mode: bit 1 the nq potentials A_q, bit 2 their gradients
// (d_j A_q at 3q + j, after the potentials); or bit 4: the curl
// u = curl A of the first three components (3 values) and, with bit 2,
// its gradient (d_j u_i at 3 + 3j + i, 12 values in all).
//
// The derivatives of the local expansion use the ladder identities of
// S_n^mu = r^n Pbar_n^|mu| e^{i mu phi} (S_n^-mu = conj S_n^mu, L_n^-mu =
// conj L_n^mu): d/dz S_n^mu = a(n,|mu|) S_{n-1}^mu, (d/dx + i d/dy) S_n^mu
// = s(mu) b(n,mu) S_{n-1}^{mu+1}, s = -1 for mu >= 0 and +1 below; each
// derivative of the expansion is an expansion of lower degree whose
// coefficient at (j, nu) is read from L at degree j+1 or j+2.
// ---------------------------------------------------------------------
// L_n^mu of one box (real-packed: n^2 for mu = 0, n^2 + 2|mu| - 1 and +1)
__device__ __forceinline__ double2 lcoef_c(const double *L, int N, int n, int mu) {
  const int am = mu < 0 ? -mu : mu;
  if (n < 0 || n > N || am > n) return make_double2(0.0, 0.0);
  if (am == 0) return make_double2(L[n * n], 0.0);
  const double re = L[n * n + 2 * am - 1], im = L[n * n + 2 * am];
  return make_double2(re, mu < 0 ? -im : im);
}

// potential, gradient (want_g) and second derivatives (want_h: xx, yy,
// zz, xy, yz, zx) of one local expansion L of order N at offset (dx, dy,
// dz) from its centre: the share of the columns k that fall to lane part of
// parts (back and forth, as in k_lap_field)
__device__ __forceinline__ void lap_local_derivs(const double *__restrict__ L, int N, double dx,
                                                 double dy, double dz, bool want_g, bool want_h,
                                                 int part, int parts,
                                                 const LapTab *__restrict__ tab, double &phi,
                                                 double g[3], double h[6]) {
  const double r = sqrt(dx * dx + dy * dy + dz * dz), rho = sqrt(dx * dx + dy * dy);
  const double Cth = r > 0.0 ? dz / r : 1.0, Sth = r > 0.0 ? rho / r : 0.0;
  const double cp = rho > 0.0 ? dx / rho : 1.0, sp = rho > 0.0 ? dy / rho : 0.0;
  double ph = 0.0, gz = 0.0, gpr = 0.0, gpi = 0.0, zz = 0.0, vr = 0.0, vi = 0.0, wr = 0.0,
         wi = 0.0;
  double pmm = 1.0 / sqrt(4.0 * kPi), rm = 1.0, cm = 1.0, sm = 0.0;
  auto lb = [&](int n, int mu) { return tab->lb[n][mu + kLapTabN]; };
  int k0 = 0;
  for (int cb = 0, odd = 0; cb <= N; cb += parts, odd ^= 1) {
    const int k = odd ? cb + parts - 1 - part : cb + part;
    if (k > N) continue;
    for (; k0 < k; k0++) {
      const int kk = k0 + 1;
      pmm *= tab->c[kk * (kk + 1) / 2 + kk].dg * Sth;
      rm *= r;
      const double tcm = cm * cp - sm * sp;
      sm = sm * cp + cm * sp;
      cm = tcm;
    }
    double p1 = 0.0, p0 = pmm, rn = rm;
    for (int j = k; j <= N; j++) {
      if (j > k) {
        const LapCol &tc = tab->c[j * (j + 1) / 2 + k];
        const double pn = Cth * tc.al * p0 - tc.be * p1;
        p1 = p0;
        p0 = pn;
        rn *= r;
      }
      // S_j^{+k} and, for k > 0, S_j^{-k} = conj
      for (int sg = 1; sg >= -1; sg -= 2) {
        if (k == 0 && sg < 0) break;
        const int nu = sg * k;
        const double Sr = rn * p0 * cm, Si = sg * rn * p0 * sm;
        auto acc = [&](double2 c, double &ore, double &oim) {
          ore += c.x * Sr - c.y * Si;
          oim += c.x * Si + c.y * Sr;
        };
        double dum = 0.0;
        acc(lcoef_c(L, N, j, nu), ph, dum);
        if (want_g) {
          const double2 cz = lcoef_c(L, N, j + 1, nu);
          const double az = tab->la[j + 1][k];
          acc(make_double2(cz.x * az, cz.y * az), gz, dum);
          const double2 cpl = lcoef_c(L, N, j + 1, nu - 1);
          const double bp = lb(j + 1, nu - 1);
          acc(make_double2(cpl.x * bp, cpl.y * bp), gpr, gpi);
        }
        if (want_h) {
          const double2 c2 = lcoef_c(L, N, j + 2, nu);
          const double f2 = tab->la[j + 2][k] * tab->la[j + 1][k];
          acc(make_double2(c2.x * f2, c2.y * f2), zz, dum);
          const int m1 = nu - 1 < 0 ? 1 - nu : nu - 1;
          const double2 cv = lcoef_c(L, N, j + 2, nu - 1);
          const double fv = tab->la[j + 2][m1] * lb(j + 1, nu - 1);
          acc(make_double2(cv.x * fv, cv.y * fv), vr, vi);
          const double2 cw = lcoef_c(L, N, j + 2, nu - 2);
          const double fw = lb(j + 2, nu - 2) * lb(j + 1, nu - 1);
          acc(make_double2(cw.x * fw, cw.y * fw), wr, wi);
        }
      }
    }
  }
  phi = ph;
  g[0] = gpr;
  g[1] = gpi;
  g[2] = gz;
  h[0] = 0.5 * (wr - zz);
  h[1] = -0.5 * (wr + zz);
  h[2] = zz;
  h[3] = 0.5 * wi;
  h[4] = vi;
  h[5] = vr;
}

// index of d_j d_k in (xx, yy, zz, xy, yz, zx)
__device__ __forceinline__ int hidx2(int j, int k) {
  if (j == k) return j;
  const int s = j + k;  // 1: xy, 3: yz, 2: zx
  return s == 1 ? 3 : (s == 3 ? 4 : 5);
}

// curl u_i = e_ikl d_k A_l and d_j u_i from the component Jacobians
// J[l][k] = d_k A_l and second derivatives H[l][.]
__device__ __forceinline__ void curl_from(const double J[3][3], const double H[3][6], bool grad,
                                          double *u) {
  u[0] += J[2][1] - J[1][2];
  u[1] += J[0][2] - J[2][0];
  u[2] += J[1][0] - J[0][1];
  if (!grad) return;
  for (int j = 0; j < 3; j++) {
    u[3 + 3 * j + 0] += H[2][hidx2(j, 1)] - H[1][hidx2(j, 2)];
    u[3 + 3 * j + 1] += H[0][hidx2(j, 2)] - H[2][hidx2(j, 0)];
    u[3 + 3 * j + 2] += H[1][hidx2(j, 0)] - H[0][hidx2(j, 1)];
  }
}

// near-field terms of one source at r = x - y (|r| above the cutoff):
// strengths sq[0..nq) (monopoles) and sd (dipoles, normal n)
__device__ __forceinline__ void near_vec(int mode, int nq, double rx, double ry, double rz,
                                         const double *sq, const double *sd, double nx,
                                         double ny, double nz, double *out) {
  const double c4 = 0.25 / kPi;
  const double r2 = rx * rx + ry * ry + rz * rz, ir = 1.0 / sqrt(r2), ir3 = ir * ir * ir,
               ir5 = ir3 * ir * ir;
  const double rv[3] = {rx, ry, rz};
  if (mode & 4) {
    // grad G = -r / (4 pi r^3); d_j grad_k G = (3 r_j r_k / r^5 - delta_jk / r^3) / (4 pi)
    const double gG[3] = {-c4 * rx * ir3, -c4 * ry * ir3, -c4 * rz * ir3};
    out[0] += gG[1] * sq[2] - gG[2] * sq[1];
    out[1] += gG[2] * sq[0] - gG[0] * sq[2];
    out[2] += gG[0] * sq[1] - gG[1] * sq[0];
    if (mode & 2)
      for (int j = 0; j < 3; j++) {
        double hG[3];
        for (int k = 0; k < 3; k++)
          hG[k] = c4 * (3.0 * rv[j] * rv[k] * ir5 - (j == k ? ir3 : 0.0));
        out[3 + 3 * j + 0] += hG[1] * sq[2] - hG[2] * sq[1];
        out[3 + 3 * j + 1] += hG[2] * sq[0] - hG[0] * sq[2];
        out[3 + 3 * j + 2] += hG[0] * sq[1] - hG[1] * sq[0];
      }
    return;
  }
  const int go = (mode & 1) ? nq : 0;
  const double nr = nx * rx + ny * ry + nz * rz;
  for (int q = 0; q < nq; q++) {
    const double qs = sq ? sq[q] * c4 : 0.0, ds = sd ? sd[q] * c4 : 0.0;
    if (mode & 1) out[q] += qs * ir + ds * nr * ir3;
    if (mode & 2) {
      out[go + 3 * q + 0] += -qs * rx * ir3 + ds * (nx * ir3 - 3.0 * nr * rx * ir5);
      out[go + 3 * q + 1] += -qs * ry * ir3 + ds * (ny * ir3 - 3.0 * nr * ry * ir5);
      out[go + 3 * q + 2] += -qs * rz * ir3 + ds * (nz * ir3 - 3.0 * nr * rz * ir5);
    }
  }
}

constexpr int kVecMaxQ = 8;    // components of the vector-source kernels
constexpr int kVecMaxOut = 32; // values per target row

__host__ __device__ __forceinline__ int vec_width(int mode, int nq) {
  if (mode & 4) return (mode & 2) ? 12 : 3;
  return ((mode & 1) ? nq : 0) + ((mode & 2) ? 3 * nq : 0);
}

// Local expansions of the target's leaf box plus the 27 neighbour boxes'
// sources (strengths nq per point, sorted order), G = 1, 4 or 16 lanes per
// target: of four lanes, lane c takes the components c, c + 4, .., the
// groups of four share each component's columns, and the sources are dealt
// as in NearSplit.  CURL apart, so that its twelve sums stay in registers.
template <bool CURL, int G>
__global__ __launch_bounds__(128) void k_lap_field_vec(
    const double *__restrict__ xt, const uint32_t *__restrict__ tid, unsigned ntgt,
    const uint32_t *__restrict__ start, const uint32_t *__restrict__ end,
    const double *__restrict__ xyz, const double *__restrict__ q,
    const double *__restrict__ nrm, const double *__restrict__ dip, int nq, int level,
    double x0, double y0, double z0, double D, int N, const double *__restrict__ mpr,
    size_t pst, int mode, double *__restrict__ f, int fstr, const LapTab *__restrict__ tab) {
  constexpr int GC = G >= 4 ? 4 : 1, GP = G / GC;  // lanes over components, over columns
  const unsigned id = blockIdx.x * blockDim.x + threadIdx.x, t = id / G;
  const int lane = (int)(id % G);
  if (t >= ntgt) return;  // the same in a group's lanes
  const double px = xt[4 * (size_t)t], py = xt[4 * (size_t)t + 1], pz = xt[4 * (size_t)t + 2];
  const uint64_t b = point_code(px, py, pz, x0, y0, z0, D) >> (3 * (20 - level));
  const int bi = compact3(b), bj = compact3(b >> 1), bk = compact3(b >> 2);
  const double w = D / (double)(1u << level);
  const double dx = px - (x0 + w * (bi + 0.5)), dy = py - (y0 + w * (bj + 0.5)),
               dz = pz - (z0 + w * (bk + 0.5));
  const size_t C = (size_t)(N + 1) * (N + 1);
  constexpr int NO = CURL ? 12 : kVecMaxOut;
  double out[NO];
#pragma unroll
  for (int i = 0; i < NO; i++) out[i] = 0.0;
  const int go = (mode & 1) ? nq : 0;
  for (int l = lane % GC; l < (CURL ? 3 : nq); l += GC) {
    double phi, g[3], h[6];
    lap_local_derivs(mpr + l * pst + b * C, N, dx, dy, dz, CURL || (mode & 2) != 0,
                     CURL && (mode & 2) != 0, lane / GC, GP, tab, phi, g, h);
    if constexpr (CURL) {
      double J[3][3], H[3][6];
#pragma unroll
      for (int c = 0; c < 3; c++) {
#pragma unroll
        for (int i = 0; i < 3; i++) J[c][i] = l == c ? g[i] : 0.0;
#pragma unroll
        for (int i = 0; i < 6; i++) H[c][i] = l == c ? h[i] : 0.0;
      }
      curl_from(J, H, (mode & 2) != 0, out);
    } else {
      if (mode & 1) out[l] += phi;
      if (mode & 2)
        for (int j = 0; j < 3; j++) out[go + 3 * l + j] += g[j];
    }
  }
  near_sources<G>(lane, bi, bj, bk, level, start, end, [&](uint32_t s) {
    const double rx = px - xyz[4 * (size_t)s], ry = py - xyz[4 * (size_t)s + 1],
                 rz = pz - xyz[4 * (size_t)s + 2];
    if (rx * rx + ry * ry + rz * rz <= 1e-12) return;
    near_vec(CURL ? 4 | (mode & 2) : mode & 3, nq, rx, ry, rz,
             q ? q + (size_t)s * nq : nullptr, dip ? dip + (size_t)s * nq : nullptr,
             dip ? nrm[4 * (size_t)s] : 0.0, dip ? nrm[4 * (size_t)s + 1] : 0.0,
             dip ? nrm[4 * (size_t)s + 2] : 0.0, out);
  });
  double *o = f + (size_t)tid[t] * fstr;
  const int nout = vec_width(mode, nq);
#pragma unroll
  for (int i = 0; i < NO; i++) {
    if (i < nout) {
      const double v = group_sum<G>(out[i]);
      if (lane == 0) o[i] += v;
    }
  }
}

// direct sums with vector sources (src/direct-laplace.c:87-198, :200-336):
// the same modes and rows as k_lap_field_vec, every source, sources
// through LDS 128 at a time; strengths nq per source (unsorted order)
__global__ __launch_bounds__(128) void k_lap_direct_vec(
    const double *__restrict__ xyz, const double *__restrict__ q,
    const double *__restrict__ nrm, const double *__restrict__ dip, int nq, unsigned nsrc,
    const double *__restrict__ xt, unsigned ntgt, int mode, double cut2,
    double *__restrict__ f, int fstr) {
  __shared__ double sx[128][4], sq[128][kVecMaxQ], sd[128][kVecMaxQ];
  const unsigned t = blockIdx.x * blockDim.x + threadIdx.x;
  double px = 0, py = 0, pz = 0;
  if (t < ntgt) {
    px = xt[4 * (size_t)t];
    py = xt[4 * (size_t)t + 1];
    pz = xt[4 * (size_t)t + 2];
  }
  double out[kVecMaxOut];
  for (int i = 0; i < kVecMaxOut; i++) out[i] = 0.0;
  for (unsigned s0 = 0; s0 < nsrc; s0 += 128) {
    const unsigned s = s0 + threadIdx.x;
    __syncthreads();
    if (s < nsrc) {
      for (int c = 0; c < 3; c++) sx[threadIdx.x][c] = xyz[4 * (size_t)s + c];
      for (int c = 0; c < nq; c++) {
        sq[threadIdx.x][c] = q ? q[(size_t)s * nq + c] : 0.0;
        sd[threadIdx.x][c] = dip ? dip[(size_t)s * nq + c] : 0.0;
      }
    }
    __syncthreads();
    const unsigned ns = nsrc - s0 < 128 ? nsrc - s0 : 128;
    for (unsigned k = 0; k < ns; k++) {
      const double rx = px - sx[k][0], ry = py - sx[k][1], rz = pz - sx[k][2];
      if (rx * rx + ry * ry + rz * rz <= cut2) continue;
      const size_t sk = s0 + k;
      near_vec(mode, nq, rx, ry, rz, q ? sq[k] : nullptr, dip ? sd[k] : nullptr,
               dip ? nrm[4 * sk] : 0.0, dip ? nrm[4 * sk + 1] : 0.0, dip ? nrm[4 * sk + 2] : 0.0,
               out);
    }
  }
  if (t >= ntgt) return;
  double *o = f + (size_t)t * fstr;
  const int nout = vec_width(mode, nq);
  for (int i = 0; i < nout; i++) o[i] += out[i];
}

// ---------------------------------------------------------------------
// FP64 direct sum, LDS-tiled (src/direct-laplace.c:200-336)
// ---------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_lap_direct(
    const double *xyz, const double *q, const double *nrm, const double *dip,
    unsigned nsrc, const double *xt, unsigned ntgt, int field, double cut2,
    double *f, int fstr) {
  __shared__ double sx[256], sy[256], sz[256], sq[256], snx[256], sny[256],
      snz[256], sd[256];
  unsigned t = blockIdx.x * blockDim.x + threadIdx.x;
  double px = 0, py = 0, pz = 0;
  if (t < ntgt) {
    px = xt[4 * (size_t)t];
    py = xt[4 * (size_t)t + 1];
    pz = xt[4 * (size_t)t + 2];
  }
  double phi = 0, gx = 0, gy = 0, gz = 0;
  for (unsigned s0 = 0; s0 < nsrc; s0 += 256) {
    unsigned s = s0 + threadIdx.x;
    __syncthreads();
    if (s < nsrc) {
      sx[threadIdx.x] = xyz[4 * (size_t)s];
      sy[threadIdx.x] = xyz[4 * (size_t)s + 1];
      sz[threadIdx.x] = xyz[4 * (size_t)s + 2];
      sq[threadIdx.x] = q ? q[s] : 0.0;
      sd[threadIdx.x] = dip ? dip[s] : 0.0;
      snx[threadIdx.x] = dip ? nrm[4 * (size_t)s] : 0.0;
      sny[threadIdx.x] = dip ? nrm[4 * (size_t)s + 1] : 0.0;
      snz[threadIdx.x] = dip ? nrm[4 * (size_t)s + 2] : 0.0;
    }
    __syncthreads();
    unsigned ns = nsrc - s0 < 256 ? nsrc - s0 : 256;
    for (unsigned k = 0; k < ns; k++) {
      double rx = px - sx[k], ry = py - sy[k], rz = pz - sz[k];
      double r2 = rx * rx + ry * ry + rz * rz;
      if (r2 <= cut2) continue;
      double ir = 1.0 / sqrt(r2), ir3 = ir * ir * ir;
      double qs = sq[k];
      phi += qs * ir;
      gx -= qs * rx * ir3;
      gy -= qs * ry * ir3;
      gz -= qs * rz * ir3;
      if (dip) {
        double nr = snx[k] * rx + sny[k] * ry + snz[k] * rz, ds = sd[k];
        double ir5 = ir3 * ir * ir;
        phi += ds * nr * ir3;
        gx += ds * (snx[k] * ir3 - 3.0 * nr * rx * ir5);
        gy += ds * (sny[k] * ir3 - 3.0 * nr * ry * ir5);
        gz += ds * (snz[k] * ir3 - 3.0 * nr * rz * ir5);
      }
    }
  }
  if (t >= ntgt) return;
  const double c4 = 0.25 / kPi;
  double *out = f + (size_t)t * fstr;
  int o = 0;
  if (field & 1) out[o++] += phi * c4;
  if (field & 2) {
    out[o++] += gx * c4;
    out[o++] += gy * c4;
    out[o++] += gz * c4;
  }
}

static inline unsigned nblk(size_t n, unsigned b) {
  return (unsigned)((n + b - 1) / b);
}

__global__ void k_d2f(const double *in, float *out, size_t n) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = (float)in[i];
}

}  // namespace wbfmm

using namespace wbfmm;

// the factors' table, built by the first call that needs it (finished
// before it is published: other streams read it then).  While the calling
// stream is captured the table is built on a stream of its own, in the
// capture mode that allows it: the field entries allocate and wait for
// nothing, and can be captured from a process's first call on.
static LapTab *g_laptab = nullptr;
static std::mutex g_laptab_mu;

static int build_lap_tab(hipStream_t s) {
  LapTab *t = nullptr;
  WBFMM_CHECK(hipMalloc((void **)&t, sizeof(LapTab)));
  hipLaunchKernelGGL(k_lap_tab, dim3(nblk(kLapTabN * (2 * kLapTabN + 1), 256)), dim3(256), 0, s, t);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) {
    (void)hipFree(t);
    return fail("factor table", e);
  }
  g_laptab = t;
  return 0;
}

static int lap_tab(const LapTab **out) {
  std::lock_guard<std::mutex> lk(g_laptab_mu);
  if (!g_laptab) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    WBFMM_CHECK(hipStreamIsCapturing(stream(), &st));
    int rc;
    if (st == hipStreamCaptureStatusNone) {
      rc = build_lap_tab(stream());
    } else {
      hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
      WBFMM_CHECK(hipThreadExchangeStreamCaptureMode(&mode));
      hipStream_t side = nullptr;
      hipError_t e = hipStreamCreateWithFlags(&side, hipStreamNonBlocking);
      rc = e == hipSuccess ? build_lap_tab(side) : fail("hipStreamCreateWithFlags", e);
      if (side) (void)hipStreamDestroy(side);
      (void)hipThreadExchangeStreamCaptureMode(&mode);
    }
    if (rc) return rc;
  }
  *out = g_laptab;
  return 0;
}

template <typename T>
static int lap_field(const char *name, const double *xt, const uint32_t *tid, unsigned n,
                     const uint32_t *start, const uint32_t *end, const double *xyz,
                     const double *q, const double *nrm, const double *dip, unsigned level,
                     const double *x0, double D, int N, double rs, const T *mpr, int field,
                     double *f, int fstr, unsigned nleaf) {
  if (N < 0 || N > kMaxN) return WBFMM_HIP_ERR_ORDER;
  if (n == 0) return 0;
  const LapTab *tab = nullptr;
  const int rc = lap_tab(&tab);
  if (rc) return rc;
#define LAP_FIELD(G)                                                                          \
  case G:                                                                                     \
    WBFMM_LAUNCH(name, (k_lap_field<T, G>), dim3(nblk((size_t)n * G, 128)), dim3(128), 0, xt, \
                 tid, n, start, end, xyz, q, nrm, dip, (int)level, x0[0], x0[1], x0[2], D, N, \
                 rs, mpr, field, f, fstr, tab);                                               \
    return 0;
  switch (wbfmm_hip_lap_field_lanes(n, nleaf)) {
    LAP_FIELD(1)
    LAP_FIELD(2)
    LAP_FIELD(4)
    LAP_FIELD(8)
    LAP_FIELD(16)
  }
#undef LAP_FIELD
  return WBFMM_HIP_ERR_ARG;
}

// one wavefront per box: groups of 16 lanes up to order 15, 32 up to 31,
// 64 above; LDS holds one expansion per group
template <typename T>
static int lap_p2m_wave(const uint32_t *boxes, unsigned nbox, const uint32_t *start,
                        const uint32_t *end, const double *xyz, const double *q,
                        const double *nrm, const double *dip, unsigned level, const double *x0,
                        double D, int N, double rs, T *mps, const char *name) {
  if (N < 0 || N > kMaxN) return WBFMM_HIP_ERR_ORDER;
  if (nbox == 0) return 0;
  const size_t C = (size_t)(N + 1) * (N + 1);
  const LapTab *tab = nullptr;
  const int rc = lap_tab(&tab);
  if (rc) return rc;
  if (N <= 15) {
    WBFMM_LAUNCH(name, (k_lap_p2m_wave<T, 16>), dim3(nbox), dim3(64), 4 * C * sizeof(double),
                 boxes, nbox, start, end, xyz, q, nrm, dip, (int)level, x0[0], x0[1], x0[2], D,
                 N, rs, mps, tab);
  } else if (N <= 31) {
    WBFMM_LAUNCH(name, (k_lap_p2m_wave<T, 32>), dim3(nbox), dim3(64), 2 * C * sizeof(double),
                 boxes, nbox, start, end, xyz, q, nrm, dip, (int)level, x0[0], x0[1], x0[2], D,
                 N, rs, mps, tab);
  } else {
    WBFMM_LAUNCH(name, (k_lap_p2m_wave<T, 64>), dim3(nbox), dim3(64), C * sizeof(double),
                 boxes, nbox, start, end, xyz, q, nrm, dip, (int)level, x0[0], x0[1], x0[2], D,
                 N, rs, mps, tab);
  }
  return 0;
}

// monopole P2M with a group of lanes per box (orders up to 16)
template <typename T>
static int lap_p2m_cols(const uint32_t *boxes, unsigned nbox, const uint32_t *start,
                        const uint32_t *end, const double *xyz, const double *q,
                        unsigned level, const double *x0, double D, int N, double rs, T *mps,
                        const char *name) {
  const int L = N / 2 + 1, per = 4 * (64 / L);  // boxes per block of four wavefronts
  const dim3 grid((nbox + per - 1) / per);
#define WBFMM_P2M_COLS(NB)                                                                 \
  WBFMM_LAUNCH(name, (k_lap_p2m_cols<T, NB>), grid, dim3(256), 0, boxes, nbox, start, end, \
               xyz, q, (int)level, x0[0], x0[1], x0[2], D, N, rs, mps)
  if (N <= 8)
    WBFMM_P2M_COLS(8);
  else if (N <= 12)
    WBFMM_P2M_COLS(12);
  else
    WBFMM_P2M_COLS(16);
#undef WBFMM_P2M_COLS
  return 0;
}

extern "C" {

int wbfmm_hip_lap_p2m(const uint32_t *boxes, unsigned nbox,
                      const uint32_t *start, const uint32_t *end,
                      const double *xyz, const double *q, const double *nrm,
                      const double *dip, unsigned level, const double *x0,
                      double D, int N, double *mps) {
  if (N < 0 || N > kMaxN) return WBFMM_HIP_ERR_ORDER;
  if (nbox == 0) return 0;
  if (!dip && q && N <= 16) return lap_p2m_cols<double>(boxes, nbox, start, end, xyz, q, level, x0, D, N,
                                             1.0, mps, "lap_p2m");
  WBFMM_LAUNCH("lap_p2m", k_lap_p2m<double>, dim3(nblk(nbox, 64)), dim3(64), 0,
               boxes, nbox, start, end, xyz, q, nrm, dip, (int)level, x0[0],
               x0[1], x0[2], D, N, 1.0, mps);
  return 0;
}

int wbfmm_hip_lap_p2m_f32(const uint32_t *boxes, unsigned nbox,
                          const uint32_t *start, const uint32_t *end,
                          const double *xyz, const double *q, const double *nrm,
                          const double *dip, unsigned level, const double *x0,
                          double D, int N, float *mps) {
  if (N < 0 || N > kMaxN) return WBFMM_HIP_ERR_ORDER;
  if (nbox == 0) return 0;
  const double w = D / (double)(1u << level);
  if (!dip && q && N <= 16) return lap_p2m_cols<float>(boxes, nbox, start, end, xyz, q, level, x0, D, N,
                                            1.0 / w, mps, "lap_p2m_f32");
  WBFMM_LAUNCH("lap_p2m_f32", k_lap_p2m<float>, dim3(nblk(nbox, 64)), dim3(64), 0,
               boxes, nbox, start, end, xyz, q, nrm, dip, (int)level, x0[0],
               x0[1], x0[2], D, N, 1.0 / w, mps);
  return 0;
}

int wbfmm_hip_lap_p2m_wave(const uint32_t *boxes, unsigned nbox, const uint32_t *start,
                           const uint32_t *end, const double *xyz, const double *q,
                           const double *nrm, const double *dip, unsigned level,
                           const double *x0, double D, int N, double *mps) {
  return lap_p2m_wave<double>(boxes, nbox, start, end, xyz, q, nrm, dip, level, x0, D, N, 1.0,
                              mps, "lap_p2m");
}

int wbfmm_hip_lap_p2m_wave_f32(const uint32_t *boxes, unsigned nbox, const uint32_t *start,
                               const uint32_t *end, const double *xyz, const double *q,
                               const double *nrm, const double *dip, unsigned level,
                               const double *x0, double D, int N, float *mps) {
  const double w = D / (double)(1u << level);
  return lap_p2m_wave<float>(boxes, nbox, start, end, xyz, q, nrm, dip, level, x0, D, N,
                             1.0 / w, mps, "lap_p2m_f32");
}

int wbfmm_hip_lap_m2m(const uint32_t *parents, unsigned npar,
                      const uint32_t *cstart, const uint32_t *cend,
                      unsigned level, double D, int Nc, int Np,
                      const double *mps_child, double *mps_parent,
                      const double *rot, const wbfmm_rot_layout_t *lay,
                      const double *coax) {
  if (Nc > lay->L || Np > lay->L || Nc > kMaxN || Np > kMaxN)
    return WBFMM_HIP_ERR_ORDER;
  if (npar == 0) return 0;
  double wc = D / (double)(1u << level);
  double t = sqrt(3.0) * 0.5 * wc;
  int Cc = (Nc + 1) * (Nc + 1), Cp = (Np + 1) * (Np + 1);
  size_t sh = sizeof(double) * (2 * Cc + Cp + Np + 1);
  const double *cf_ss = coax;  // kind 0
  WBFMM_LAUNCH("lap_m2m", k_lap_m2m, dim3(npar), dim3(64), sh, parents, npar,
               cstart, cend, t, Nc, Np, mps_child, mps_parent,
               rot + lay->up_fwd, rot + lay->up_back, lay->nrot, cf_ss,
               lay->L);
  return 0;
}

int wbfmm_hip_lap_m2l(const uint32_t *targets, unsigned ntgt,
                      const uint32_t *sstart, const uint32_t *send,
                      unsigned level, double D, int Ns, int Nr,
                      const double *mps, double *mpr, const double *rot,
                      const wbfmm_rot_layout_t *lay, const double *coax) {
  if (Ns > lay->L || Nr > lay->L || Ns > kMaxN || Nr > kMaxN)
    return WBFMM_HIP_ERR_ORDER;
  if (ntgt == 0) return 0;
  double w = D / (double)(1u << level);
  int Cs = (Ns + 1) * (Ns + 1), Cr = (Nr + 1) * (Nr + 1);
  size_t sh = sizeof(double) * (2 * Cs + Cr + Ns + Nr + 2);
  size_t L1 = (size_t)(lay->L + 1);
  const double *cf_sr = coax + 2 * L1 * L1 * L1;
  // the offset lengths live in the layout struct on the host; pass a
  // device copy kept at the end of the rotation block
  const double *roff = rot + lay->total;
  WBFMM_LAUNCH("lap_m2l", k_lap_m2l, dim3(ntgt), dim3(64), sh, targets, ntgt,
               sstart, send, (int)level, w, Ns, Nr, mps, mpr,
               rot + lay->m2l_fwd, rot + lay->m2l_back, lay->nrot, roff,
               cf_sr, lay->L);
  return 0;
}

int wbfmm_hip_lap_l2l(const uint32_t *parents, unsigned npar,
                      const uint32_t *cflag, unsigned level, double D,
                      int Np, int Nc, const double *mpr_parent,
                      double *mpr_child, const double *rot,
                      const wbfmm_rot_layout_t *lay, const double *coax) {
  if (Nc > lay->L || Np > lay->L || Nc > kMaxN || Np > kMaxN)
    return WBFMM_HIP_ERR_ORDER;
  if (npar == 0) return 0;
  double wc = D / (double)(1u << (level + 1));
  double t = sqrt(3.0) * 0.5 * wc;
  int Cc = (Nc + 1) * (Nc + 1), Cp = (Np + 1) * (Np + 1);
  size_t sh = sizeof(double) * (2 * Cp + Cc + Np + 1);
  size_t L1 = (size_t)(lay->L + 1);
  const double *cf_rr = coax + L1 * L1 * L1;
  WBFMM_LAUNCH("lap_l2l", k_lap_l2l, dim3(npar), dim3(64), sh, parents, npar,
               cflag, t, Np, Nc, mpr_parent, mpr_child, rot + lay->dn_fwd,
               rot + lay->dn_back, lay->nrot, cf_rr, lay->L);
  return 0;
}

// Occupied leaves of fewer than two targets on average: mostly expansion
// steps, whose scattered coefficient reads four lanes of a target share.
// Measured with one lane, two and four, orders 12 (FP64) and 9 (FP32), ms,
// at targets per occupied leaf: 1.26 (1e6 in a cube, depth 7) 2.41 1.80 1.58
// and 1.08 0.77 0.73; 1.68 (3e5, depth 6) 0.55 0.41 0.39 and 0.27 0.24 0.23;
// 1.96 0.65 0.48 0.47 and 0.37 0.31 0.29; 2.56 (6e5, depth 6) 0.80 0.67 0.75
// and 0.46 0.47 0.48; 4.9 (3e5 on a sphere, depth 7) 0.31 0.34 0.41 and 0.27
// 0.28 0.30; 14.7 (1e6 on a sphere, depth 7) 1.22 1.58 1.97 and 1.05 1.40
// 1.63.  The empty boxes of a level do not count: over all boxes the last
// two have 0.14 and 0.48 targets a leaf.
int wbfmm_hip_lap_field_lanes(unsigned n, unsigned nleaf) {
  if (n > (1u << 26)) return 1;
  const int g = field_lanes(n);
  return g < 4 && n >> 1 < nleaf ? 4 : g;
}

int wbfmm_hip_lap_field_leaves(const double *xt, const uint32_t *tid, unsigned n, unsigned nleaf,
                               const uint32_t *start, const uint32_t *end, const double *xyz,
                               const double *q, const double *nrm, const double *dip,
                               unsigned level, const double *x0, double D, int N, int f32,
                               const void *mpr, int field, double *f, int fstr) {
  const double w = D / (double)(1u << level);
  if (f32)
    return lap_field<float>("lap_l2p_p2p_f32", xt, tid, n, start, end, xyz, q, nrm, dip, level, x0,
                            D, N, 1.0 / w, (const float *)mpr, field, f, fstr, nleaf);
  return lap_field<double>("lap_l2p_p2p", xt, tid, n, start, end, xyz, q, nrm, dip, level, x0, D, N,
                           1.0, (const double *)mpr, field, f, fstr, nleaf);
}

// boxes of a level, as many as the type holds
static unsigned level_boxes(unsigned level) { return level <= 10 ? 1u << (3 * level) : ~0u; }

int wbfmm_hip_lap_field(const double *xt, const uint32_t *tid, unsigned n,
                        const uint32_t *start, const uint32_t *end,
                        const double *xyz, const double *q, const double *nrm,
                        const double *dip, unsigned level, const double *x0,
                        double D, int N, const double *mpr, int field,
                        double *f, int fstr) {
  return wbfmm_hip_lap_field_leaves(xt, tid, n, level_boxes(level), start, end, xyz, q, nrm, dip,
                                    level, x0, D, N, 0, mpr, field, f, fstr);
}

int wbfmm_hip_lap_field_f32(const double *xt, const uint32_t *tid, unsigned n,
                            const uint32_t *start, const uint32_t *end,
                            const double *xyz, const double *q, const double *nrm,
                            const double *dip, unsigned level, const double *x0,
                            double D, int N, const float *mpr, int field,
                            double *f, int fstr) {
  return wbfmm_hip_lap_field_leaves(xt, tid, n, level_boxes(level), start, end, xyz, q, nrm, dip,
                                    level, x0, D, N, 1, mpr, field, f, fstr);
}

int wbfmm_hip_to_f32(const double *in, float *out, size_t n) {
  if (n == 0) return 0;
  WBFMM_LAUNCH("to_f32", k_d2f, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, in, out, n);
  return 0;
}

int wbfmm_hip_lap_field_vec(const double *xt, const uint32_t *tid, unsigned n,
                            const uint32_t *start, const uint32_t *end, const double *xyz,
                            const double *q, const double *nrm, const double *dip, int nq,
                            unsigned level, const double *x0, double D, int N,
                            const double *mpr, size_t plane_stride, int mode, double *f,
                            int fstr) {
  if (N < 0 || N > kMaxN) return WBFMM_HIP_ERR_ORDER;
  if (nq < 1 || nq > kVecMaxQ || ((mode & 4) && nq < 3) || !(mode & 7) ||
      vec_width(mode, nq) > kVecMaxOut || fstr < vec_width(mode, nq) || ((mode & 4) && dip))
    return WBFMM_HIP_ERR_ARG;
  if (n == 0) return 0;
  const LapTab *tab = nullptr;
  const int rc = lap_tab(&tab);
  if (rc) return rc;
  const int g = n > (1u << 26) ? 1 : field_lanes(n);
#define LAP_VEC(CU, G)                                                                        \
  WBFMM_LAUNCH("lap_l2p_p2p_vec", (k_lap_field_vec<CU, G>), dim3(nblk((size_t)n * G, 128)),   \
               dim3(128), 0, xt, tid, n, start, end, xyz, q, nrm, dip, nq, (int)level, x0[0], \
               x0[1], x0[2], D, N, mpr, plane_stride, mode, f, fstr, tab)
  if (mode & 4) {
    if (g >= 16) LAP_VEC(true, 16);
    else if (g >= 4) LAP_VEC(true, 4);
    else LAP_VEC(true, 1);
  } else {
    if (g >= 16) LAP_VEC(false, 16);
    else if (g >= 4) LAP_VEC(false, 4);
    else LAP_VEC(false, 1);
  }
#undef LAP_VEC
  return 0;
}

int wbfmm_hip_lap_direct_vec(const double *xyz, const double *q, const double *nrm,
                             const double *dip, int nq, unsigned nsrc, const double *xt,
                             unsigned ntgt, int mode, double cutoff, double *f, int fstr) {
  if (nq < 1 || nq > kVecMaxQ || ((mode & 4) && nq < 3) || !(mode & 7) ||
      vec_width(mode, nq) > kVecMaxOut || fstr < vec_width(mode, nq) || ((mode & 4) && dip))
    return WBFMM_HIP_ERR_ARG;
  if (ntgt == 0) return 0;
  WBFMM_LAUNCH("lap_direct_vec", k_lap_direct_vec, dim3(nblk(ntgt, 128)), dim3(128), 0, xyz, q,
               nrm, dip, nq, nsrc, xt, ntgt, mode, cutoff * cutoff, f, fstr);
  return 0;
}

int wbfmm_hip_lap_direct(const double *xyz, const double *q,
                         const double *nrm, const double *dip, unsigned nsrc,
                         const double *xt, unsigned ntgt, int field,
                         double cutoff, double *f, int fstr) {
  if (ntgt == 0) return 0;
  WBFMM_LAUNCH("lap_direct", k_lap_direct, dim3(nblk(ntgt, 256)), dim3(256),
               0, xyz, q, nrm, dip, nsrc, xt, ntgt, field, cutoff * cutoff,
               f, fstr);
  return 0;
}

}  // extern "C"
