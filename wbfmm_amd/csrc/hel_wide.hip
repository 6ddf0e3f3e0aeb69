// hel_wide.hip -- Helmholtz M2L, M2M and L2L on FP64 matrix cores with the
// order as a run-time value: orders 28..40, whose exchange buffer does not
// fit the kernels of hel_m2l_impl.h, and levels whose two orders differ.
//
// The algebra is that of hel_m2l_mfma.hip: with the phase-rotated
// x'_m = e^{i m chi} x_m, P_m = x'_m + x'_{-m} and Q_m = x'_m - x'_{-m}
// pass through rotation, coaxial shift and rotation back separately.  That
// separation sets the layout here:
//   - a block takes one of the two through all three stages, then the
//     other, so that the exchange buffer holds (N+1)(N+2)/2 rows of 16
//     columns instead of (N+1)^2, without rows of padding (block rows are
//     consecutive; a tile's last k-step may read up to three rows of its
//     neighbour against zeros of the table).  At order 31 both copies of a
//     double buffer fit 160 KB (one barrier per stage); above, one copy.
//   - the 16 columns are 8 targets (parents) x real / imaginary part; the
//     complex coaxial stage takes a second product on the partner column.
//   - eight wavefronts share the row tiles of a stage, dealt in order of
//     their k-steps.  A tile's k-step count (at most 11) selects
//     straight-line code.  Sixteen wavefronts (128 registers each) spilled
//     312 registers at order 31.
//   - the local expansions stay in registers over all offsets, lane
//     (group, column) of wavefront w owning the units group + 4 w + 32 i.
// Bound: FP64 matrix cores, with 72 % of the tiles' entries used at order
// 30 (1744 products of 64 cycles per 8 targets and offset), and the waits
// for operands between barriers with two wavefronts per SIMD.
//
// A 3e4-point cube at depth 3, k = 8, orders 30 (tol 1e-8): M2L 63.8 ms
// (one wavefront per target on the vector unit) -> 3.6 ms, M2M and L2L 2.0
// -> 0.06 ms each, the solve 71.4 -> 7.6 ms.

#include <cstdio>

#include <hip/hip_runtime.h>

#include "hip_common.h"
#include "m2l_mfma.h"

namespace wbfmm {

constexpr int kWideW = 8;  // wavefronts per block (two of the plan's 16 lists each)

template <int NMAX>
struct WideShape {
  static constexpr int NU = (NMAX + 1) * (NMAX + 2) / 2;
  // three rows that a last k-step may read past the blocks, and the row
  // that takes a tile's unused rows
  static constexpr int ROWS = NU + 4;
  static constexpr bool DB = 2 * ROWS * 16 * (int)sizeof(double) <= 140 * 1024;
  static constexpr int NAW = (NU + 4 * kWideW - 1) / (4 * kWideW);  // units per lane
  static constexpr int NT = NMAX <= 24 ? 32 : NMAX <= 31 ? 44 : 72;  // row tiles of a part
  // the next step's sources held during the Q part, where registers allow
  static constexpr bool PRE = NMAX <= 24;
  static constexpr int TW = 2 * ((NT + 15) / 16);              // tiles per wavefront
};

// one row tile of a stage: NK k-steps of the table a (and ai on the partner
// column: the imaginary part of a complex table), four k-steps' operands
// requested at a time
template <int NK, bool CX>
__device__ __forceinline__ d4 wide_tile(const double *__restrict__ a,
                                        const double *__restrict__ ai, const double *R, int lane,
                                        double sg) {
  constexpr int ST = CX ? 4 : 8;
  d4 r4 = {0.0, 0.0, 0.0, 0.0}, i4 = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int j0 = 0; j0 < NK; j0 += ST) {
    double av[ST], bv[ST], aw[ST], bw[ST];
#pragma unroll
    for (int j = 0; j < ST && j0 + j < NK; j++) {
      av[j] = a[(j0 + j) * 64 + lane];
      if constexpr (CX) aw[j] = ai[(j0 + j) * 64 + lane];
    }
#pragma unroll
    for (int j = 0; j < ST && j0 + j < NK; j++) {
      bv[j] = R[(j0 + j) * 64 + lane];
      if constexpr (CX) bw[j] = R[(j0 + j) * 64 + (lane ^ 1)];
    }
#pragma unroll
    for (int j = 0; j < ST && j0 + j < NK; j++) {
      r4 = MF<double>::mma(av[j], bv[j], r4);
      if constexpr (CX) i4 = MF<double>::mma(aw[j], bw[j], i4);
    }
  }
  if constexpr (CX) return r4 + sg * i4;
  return r4;
}

template <int NMAX, bool CX>
__device__ __forceinline__ d4 wide_tile_n(int nk, const double *a, const double *ai,
                                          const double *R, int lane, double sg) {
  // k-steps of the largest block of each range of orders: 7, 8, 11
  switch (nk) {
#define WIDE_CASE(K)                                                    \
  case K:                                                               \
    if constexpr (K <= (NMAX + 4) / 4) return wide_tile<K, CX>(a, ai, R, lane, sg); \
    break;
    WIDE_CASE(1)
    WIDE_CASE(2)
    WIDE_CASE(3)
    WIDE_CASE(4)
    WIDE_CASE(5)
    WIDE_CASE(6)
    WIDE_CASE(7)
    WIDE_CASE(8)
    WIDE_CASE(9)
    WIDE_CASE(10)
    WIDE_CASE(11)
#undef WIDE_CASE
  }
  return d4{0.0, 0.0, 0.0, 0.0};
}

struct Real {
  static constexpr bool value = false;
};
struct Cplx {
  static constexpr bool value = true;
};

// MODE 0: M2M (sum over the occupied children of 8 parents, the parents
// overwritten; with nsplit = 8, blockIdx.y one child digit and the partial
// sums to `part'); 1: L2L (one child of 8 parents, blockIdx.y the child's
// digit, added); 2: M2L (8 targets of one Morton class, added, or the
// partial sums of split `split' of nsplit)
template <int MODE, int NMAX>
__global__ __launch_bounds__(64 * kWideW) void k_hel_wide(
    const uint32_t *__restrict__ list, unsigned nlist, ClassArgs ca,
    const uint32_t *__restrict__ cstart, const uint32_t *__restrict__ cend,
    const uint32_t *__restrict__ cflag, const uint32_t *__restrict__ occ, int level, int Nin,
    int Nout, const double2 *__restrict__ in, double2 *__restrict__ out,
    const wbfmm_hel_wide_plan_t *__restrict__ P, const double *__restrict__ A,
    const double *__restrict__ A2, const double *__restrict__ CS, int nsplit,
    double2 *__restrict__ part, unsigned ntot) {
  using SH = WideShape<NMAX>;
  constexpr int NAW = SH::NAW, W = kWideW, ROWS = SH::ROWS;
  constexpr bool DB = SH::DB;
  __shared__ double R[(DB ? 2 : 1) * ROWS * 16];
  __shared__ uint16_t maps[3][2][16 * SH::NT];
  __shared__ int2 uinf[SH::NU];  // n | m << 16, slot in P | slot in Q << 16
  __shared__ double2 cs[2][NMAX + 1];
  __shared__ unsigned vm[8][7];
  __shared__ unsigned anym[7];

  const int tid = threadIdx.x, lane = tid & 63, col = lane & 15, grp = lane >> 4, sp = col & 1;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int N = P->N, NU = P->NU, KT = P->KT, dump = ROWS - 1;
  const int Cin = (Nin + 1) * (Nin + 1), Cout = (Nout + 1) * (Nout + 1);
  double *R1 = R + (DB ? ROWS * 16 : 0);

  for (int pt = 0; pt < 2; pt++)
    for (int i = tid; i < 16 * P->nt[pt]; i += 64 * W) {
      const int m1 = P->map1[pt][i], m2 = P->map2[pt][i], m3 = P->map3[pt][i];
      maps[0][pt][i] = (uint16_t)(m1 < 0 ? dump : m1);
      maps[1][pt][i] = (uint16_t)(m2 < 0 ? dump : m2);
      maps[2][pt][i] = (uint16_t)(m3 < 0 ? dump : m3);
    }
  // unit u = (n, m): degree, order, its slots in P and Q
  for (int u = tid; u < NU; u += 64 * W) {
    int n = 0;
    while ((n + 1) * (n + 2) / 2 <= u) n++;
    uinf[u] = make_int2(n | (u - n * (n + 1) / 2) << 16, P->s1[0][u] | P->s1[1][u] << 16);
  }
  for (int i = tid; i < (DB ? 2 : 1) * ROWS * 16; i += 64 * W) R[i] = 0.0;
  for (int i = tid; i < 8 * 7; i += 64 * W) vm[i / 7][i % 7] = 0u;

  // the block's 8 targets (parents): this lane's is tg
  const int tg = col >> 1;
  int c = 0, split = MODE == 0 ? (int)blockIdx.y : 0;
  unsigned row8;
  bool tvalid;
  uint32_t tb;
  if constexpr (MODE == 2) {
    split = (int)(blockIdx.x % (unsigned)nsplit);
    const unsigned nch = ca.chunk_prefix[8], bid = blockIdx.x / (unsigned)nsplit, q8 = nch / 8;
    const unsigned chunk = bid < 8 * q8 ? (bid & 7) * q8 + (bid >> 3) : bid;
    while (c < 7 && chunk >= ca.chunk_prefix[c + 1]) c++;
    const unsigned k8 = (chunk - ca.chunk_prefix[c]) * 8 + tg;
    tvalid = k8 < ca.count[c];
    row8 = ca.start[c] + k8;
  } else {
    row8 = blockIdx.x * 8 + tg;
    tvalid = row8 < nlist;
  }
  tb = tvalid ? list[row8] : 0u;
  const int px = c & 1, py = (c >> 1) & 1, pz = (c >> 2) & 1;
  __syncthreads();

  // the sources of each target: bit k of vm[target] for step k (an offset
  // of the 6 x 6 x 6 cube, or a child digit)
  if (sp == 0) {
    if constexpr (MODE == 2) {
      const int nbox = 1 << level;
      const int ti = compact3(tb), tj = compact3(tb >> 1), tk = compact3(tb >> 2);
      for (int k = grp + 4 * wv; k < 216; k += 4 * W) {
        if (nsplit > 1 && k % nsplit != split) continue;
        const int dx = k % 6 - 2 - px, dy = (k / 6) % 6 - 2 - py, dz = k / 36 - 2 - pz;
        if (dx >= -1 && dx <= 1 && dy >= -1 && dy <= 1 && dz >= -1 && dz <= 1) continue;
        const int si = ti + dx, sj = tj + dy, sk = tk + dz;
        if (!tvalid || si < 0 || si >= nbox || sj < 0 || sj >= nbox || sk < 0 || sk >= nbox)
          continue;
        const uint64_t sb = spread3(si) | (spread3(sj) << 1) | (spread3(sk) << 2);
        if ((occ[sb >> 5] >> (sb & 31)) & 1u) atomicOr(&vm[tg][k >> 5], 1u << (k & 31));
      }
    } else if (wv == 0 && grp == 0 && tvalid) {
      unsigned m = 0;
      for (int cc = 0; cc < 8; cc++) {
        const uint64_t cb = 8 * (uint64_t)tb + cc;
        if (MODE == 0 ? cend[cb] > cstart[cb] && (nsplit == 1 || cc == (int)blockIdx.y)
                      : cc == (int)blockIdx.y && (!cflag || cflag[cb] != 0))
          m |= 1u << cc;
      }
      vm[tg][0] = m;
    }
  }
  __syncthreads();
  if (tid < 7) {
    unsigned a = 0;
    for (int j = 0; j < 8; j++) a |= vm[j][tid];
    anym[tid] = a;
  }
  __syncthreads();

  unsigned am[7];
#pragma unroll
  for (int w = 0; w < 7; w++) am[w] = __builtin_amdgcn_readfirstlane(anym[w]);
  constexpr int kEnd = 216;
  auto next_k = [&](int k) {
    int kn = k + 1;
#pragma unroll
    for (int w = 0; w < 7; w++) {
      if (kn < 32 * (w + 1)) {
        const unsigned bits = am[w] & (kn > 32 * w ? ~0u << (kn - 32 * w) : ~0u);
        if (bits) return 32 * w + (int)__builtin_ctz(bits);
        kn = 32 * (w + 1);
      }
    }
    return kEnd;
  };

  const int ubase = grp + 4 * wv;
  double pre_re[NAW], pre_im[NAW], qh[NAW];
  // x_{+m} on the real lane, x_{-m} on the imaginary one (zero for a
  // target without this source, and above the source's order); every
  // wavefront writes the step's phases (the same values)
  auto load_sources = [&](int k, int p, const int2 *ui) {
    const bool v = (vm[tg][k >> 5] >> (k & 31)) & 1u;
    uint32_t sb = tb;
    int crow = k;
    if constexpr (MODE == 2) {
      const int dx = k % 6 - 2 - px, dy = (k / 6) % 6 - 2 - py, dz = k / 36 - 2 - pz;
      sb = morton_add(tb, dilate_offset(dx, 0, kMortonX), dilate_offset(dy, 1, kMortonY),
                      dilate_offset(dz, 2, kMortonZ));
      crow = (dx + 3) * 49 + (dy + 3) * 7 + dz + 3;
    }
    const double2 *src = in + (MODE == 0 ? 8 * (uint64_t)tb + k : (uint64_t)sb) * Cin;
    if (lane <= N) {
      const double *t = CS + ((size_t)crow * (N + 1) + lane) * 2;
      cs[p][lane] = make_double2(t[0], t[1]);
    }
#pragma unroll
    for (int i = 0; i < NAW; i++) {
      const int u = ubase + 4 * W * i;
      pre_re[i] = pre_im[i] = 0.0;
      if (u < NU && v) {
        const int nm = ui[u].x, n = nm & 0xffff, m = nm >> 16;
        if (n <= Nin) {
          const double2 q = src[n * (n + 1) + (sp ? -m : m)];
          pre_re[i] = q.x;
          pre_im[i] = q.y;
        }
      }
    }
  };
  // x'_{+-m} = e^{+-i m chi} x_{+-m}; the partner lane holds the other
  // sign.  P goes into R, Q stays in the lane until its turn
  auto deposit_p = [&](int p, const int2 *ui) {
#pragma unroll
    for (int i = 0; i < NAW; i++) {
      const int u = ubase + 4 * W * i;
      const int2 inf = ui[u < NU ? u : NU - 1];
      const double2 e = cs[p][inf.x >> 16];
      const double es = sp ? -e.y : e.y;
      const double xr = e.x * pre_re[i] - es * pre_im[i];
      const double xi = es * pre_re[i] + e.x * pre_im[i];
      const double yr = __shfl_xor(xr, 1), yi = __shfl_xor(xi, 1);
      qh[i] = sp ? yi - xi : xr - yr;
      if (u < NU) R[(inf.y & 0xffff) * 16 + col] = sp ? yi + xi : xr + yr;
    }
  };
  auto deposit_q = [&](const int2 *ui) {
#pragma unroll
    for (int i = 0; i < NAW; i++) {
      const int u = ubase + 4 * W * i;
      if (u >= NU) continue;
      const int2 inf = ui[u];
      if (inf.x >> 16) R[(inf.y >> 16) * 16 + col] = qh[i];
    }
  };
  const double sg = sp ? 1.0 : -1.0;
  // one stage of part pt with table a (ai: the imaginary part of a complex
  // table), rows sent through map mi.  Double-buffered: Ri -> Ro, one
  // barrier; single: results held in registers between two barriers
  auto stage = [&](auto cxc, int pt, const double *a, const double *ai, const double *Ri,
                   double *Ro, int mi) {
    constexpr bool CX = decltype(cxc)::value;
    const int t0 = P->wbeg[pt][2 * wv], t1 = P->wbeg[pt][2 * wv + 2];
    const uint16_t *mp = maps[mi][pt];
    auto put = [&](int t, const d4 &y) {
#pragma unroll
      for (int q = 0; q < 4; q++) Ro[mp[16 * t + MF<double>::drow(grp, q)] * 16 + col] = y[q];
    };
    auto product = [&](int t) {
      const int nk = P->tile[pt][t][1], ko = P->tile[pt][t][2];
      return wide_tile_n<NMAX, CX>(nk, a + (size_t)ko * 64, ai + (size_t)ko * 64,
                                   Ri + P->tile[pt][t][0] * 16, lane, sg);
    };
    if constexpr (DB) {
      for (int t = t0; t < t1; t++) put(t, product(t));
      __syncthreads();
    } else {
      d4 y[SH::TW];
#pragma unroll
      for (int i = 0; i < SH::TW; i++)
        if (t0 + i < t1) y[i] = product(t0 + i);
      __syncthreads();
#pragma unroll
      for (int i = 0; i < SH::TW; i++)
        if (t0 + i < t1) put(t0 + i, y[i]);
      __syncthreads();
    }
  };
  auto stages = [&](int pt, const double *ar, const double *ac, const double *aci) {
    stage(Real{}, pt, ar, ar, R, R1, 0);
    if constexpr (MODE == 2)
      stage(Cplx{}, pt, ac, aci, R1, R, 1);
    else
      stage(Real{}, pt, ac, ac, R1, R, 1);
    stage(Real{}, pt, ar, ar, R, R1, 2);
  };

  double acc_re[NAW], acc_im[NAW];
#pragma unroll
  for (int i = 0; i < NAW; i++) acc_re[i] = acc_im[i] = 0.0;
  // y_{+-nu} = (P +- Q)/2 (y_0 = P/2), then L^{+-nu} += e^{-+i nu chi} y:
  // this part's half of it
  auto gather = [&](int pt, int p, const int2 *ui) {
    const double h = pt && sp ? -0.5 : 0.5;
    const int c0 = col & ~1;
#pragma unroll
    for (int i = 0; i < NAW; i++) {
      const int u = ubase + 4 * W * i;
      if (u >= NU) continue;
      const int nu = ui[u].x >> 16;
      if (pt && !nu) continue;
      const double2 e = cs[p][nu];
      const double es = sp ? -e.y : e.y;
      const double yr = h * R1[u * 16 + c0], yi = h * R1[u * 16 + c0 + 1];
      acc_re[i] += e.x * yr + es * yi;
      acc_im[i] += e.x * yi - es * yr;
    }
    if constexpr (!DB) __syncthreads();  // every read of R done before the next deposit
  };
  auto table_of = [&](int k, int &th, int &ri) {
    if constexpr (MODE == 2) {
      const int dx = k % 6 - 2 - px, dy = (k / 6) % 6 - 2 - py, dz = k / 36 - 2 - pz;
      const int o = (dx + 3) * 49 + (dy + 3) * 7 + dz + 3;
      th = __builtin_amdgcn_readfirstlane(P->th[o]);
      ri = __builtin_amdgcn_readfirstlane(P->rix[o]);
    } else {
      th = MODE == 0 ? (k >> 2) & 1 : 1 - ((k >> 2) & 1);
      ri = 0;
    }
  };

  int k = __builtin_amdgcn_readfirstlane(next_k(-1)), p = 0;
  if (k < kEnd) {
    load_sources(k, 0, uinf);
    deposit_p(0, uinf);
  }
  __syncthreads();
  while (k < kEnd) {
    // z0 keeps the units' records from being held in registers over the loop
    int z0, th, ri;
    asm volatile("s_mov_b32 %0, 0" : "=s"(z0));
    const int2 *ui = uinf + z0;
    table_of(k, th, ri);
    const int kn = __builtin_amdgcn_readfirstlane(next_k(k));
    const double *ar = A + (size_t)th * KT * 64;
    const double *ac = A2 + (size_t)(MODE == 2 ? 2 * ri : 0) * KT * 64;
    const double *aci = ac + (MODE == 2 ? (size_t)KT * 64 : 0);
    stages(0, ar, ac, aci);
    gather(0, p, ui);
    deposit_q(ui);
    __syncthreads();
    if (SH::PRE && kn < kEnd) load_sources(kn, p ^ 1, ui);
    stages(1, ar, ac, aci);
    gather(1, p, ui);
    if (kn < kEnd) {
      if (!SH::PRE) load_sources(kn, p ^ 1, ui);
      deposit_p(p ^ 1, ui);
    }
    __syncthreads();
    p ^= 1;
    k = kn;
  }

  bool store = tvalid;
  if constexpr (MODE == 1) store = store && ((vm[tg][0] >> blockIdx.y) & 1u);
  if (!store) return;
  double2 *dst = MODE == 1   ? out + (8 * (uint64_t)tb + blockIdx.y) * Cout
                 : nsplit > 1 ? part + ((size_t)split * ntot + row8) * Cout
                              : out + (uint64_t)tb * Cout;
#pragma unroll
  for (int i = 0; i < NAW; i++) {
    const int u = ubase + 4 * W * i;
    if (u >= NU) continue;
    const int n = uinf[u].x & 0xffff, m = uinf[u].x >> 16;
    if (n > Nout || (sp && m == 0)) continue;  // L^0 is the real lane's
    const int r = n * (n + 1) + (sp ? -m : m);
    if (MODE == 0 || nsplit > 1) {
      dst[r] = make_double2(acc_re[i], acc_im[i]);
    } else {
      const double2 o = dst[r];
      dst[r] = make_double2(o.x + acc_re[i], o.y + acc_im[i]);
    }
  }
}

// parent i = the sum of its children's parts, in child order
__global__ void k_wide_m2m_sum(const uint32_t *__restrict__ parents, unsigned npar, int C,
                               const double2 *__restrict__ part, double2 *__restrict__ out) {
  const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (size_t)npar * C) return;
  double2 s = part[e];
  for (int c = 1; c < 8; c++) {
    const double2 v = part[(size_t)c * npar * C + e];
    s = make_double2(s.x + v.x, s.y + v.y);
  }
  out[(size_t)parents[e / C] * C + e % C] = s;
}

template <int MODE>
static int launch_wide(const char *name, dim3 grid, const uint32_t *list, unsigned nlist,
                       const ClassArgs &ca, const uint32_t *cstart, const uint32_t *cend,
                       const uint32_t *cflag, const uint32_t *occ, int level, int Nin, int Nout,
                       const double *in, double *out, const void *plan_dev, const double *A,
                       const double *A2, const double *CS, int nsplit, double *part,
                       unsigned ntot, const wbfmm_hel_wide_plan_t *hp) {
#define WIDE_LAUNCH(NM)                                                                       \
  WBFMM_LAUNCH(name, (k_hel_wide<MODE, NM>), grid, dim3(64 * kWideW), 0, list, nlist, ca,     \
               cstart, cend, cflag, occ, level, Nin, Nout, (const double2 *)in,               \
               (double2 *)out, (const wbfmm_hel_wide_plan_t *)plan_dev, A, A2, CS, nsplit,    \
               (double2 *)part, ntot)
  const int nt = hp->nt[0] > hp->nt[1] ? hp->nt[0] : hp->nt[1];
  if (hp->N <= 24 && nt <= WideShape<24>::NT)
    WIDE_LAUNCH(24);
  else if (hp->N <= 31 && nt <= WideShape<31>::NT)
    WIDE_LAUNCH(31);
  else if (hp->N <= 40 && nt <= WideShape<40>::NT)
    WIDE_LAUNCH(40);
  else
    return WBFMM_HIP_ERR_ORDER;
#undef WIDE_LAUNCH
  return 0;
}

}  // namespace wbfmm

using namespace wbfmm;

extern "C" {

int wbfmm_hip_hel_wide_m2l(const uint32_t *cls, const unsigned *cstart, const unsigned *ccount,
                           const uint32_t *sstart, const uint32_t *send, unsigned level, int Ns,
                           int Nr, const double *mps, double *mpr, const void *plan_dev,
                           const double *A, const double *A2, const double *CS,
                           const wbfmm_hel_wide_plan_t *plan_host) {
  ClassArgs ca;
  ca.qc = 0;
  unsigned nch = 0, ntot = 0;
  for (int c = 0; c < 8; c++) {
    ca.start[c] = cstart[c];
    ca.count[c] = ccount[c];
    ca.chunk_prefix[c] = nch;
    nch += (ccount[c] + 7) / 8;
    ntot += ccount[c];
  }
  ca.chunk_prefix[8] = nch;
  if (nch == 0) return 0;
  // source boxes are found by 30-bit Morton arithmetic
  if (level < 2 || level > (unsigned)kMortonAddMaxLevel) return WBFMM_HIP_ERR_ARG;
  if (!plan_host || plan_host->N != (Ns > Nr ? Ns : Nr)) return WBFMM_HIP_ERR_ARG;
  uint32_t *occ = nullptr;
  {
    const int ro = occupancy_bits(sstart, send, level, &occ);
    if (ro) return ro;
  }
  const int nsplit = wide_nsplit(nch);
  const size_t C = (size_t)(Nr + 1) * (Nr + 1);
  double *part = nullptr;
  if (nsplit > 1 && dmalloc((void **)&part, sizeof(double) * 2 * (size_t)nsplit * ntot * C)) {
    dfree(occ);
    return WBFMM_HIP_ERR_NOMEM;
  }
  const int rc = launch_wide<2>("hel_m2l", dim3(nch * nsplit), cls, ntot, ca, nullptr, nullptr,
                                nullptr, occ, (int)level, Ns, Nr, mps, mpr, plan_dev, A, A2, CS,
                                nsplit, part, ntot, plan_host);
  if (!rc && nsplit > 1) {
    const size_t ne = (size_t)ntot * 2 * C;
    WBFMM_LAUNCH("m2l_reduce", k_m2l_reduce<double>, dim3((unsigned)((ne + 255) / 256)),
                 dim3(256), 0, cls, ntot, nsplit, (int)(2 * C), (const double *)part, mpr);
  }
  dfree(part);
  dfree(occ);
  return rc;
}

int wbfmm_hip_hel_wide_shift(int mode, const uint32_t *parents, unsigned npar,
                             const uint32_t *cstart, const uint32_t *cend,
                             const uint32_t *cflag, int Nin, int Nout, const double *in,
                             double *out, const void *plan_dev, const double *A,
                             const double *A2, const double *CS,
                             const wbfmm_hel_wide_plan_t *plan_host) {
  if (npar == 0) return 0;
  if (mode != 0 && mode != 1) return WBFMM_HIP_ERR_ARG;
  if (mode == 0 && (!cstart || !cend)) return WBFMM_HIP_ERR_ARG;
  if (!plan_host || plan_host->N != (Nin > Nout ? Nin : Nout)) return WBFMM_HIP_ERR_ARG;
  ClassArgs ca{};
  const unsigned nb = (npar + 7) / 8;
  if (mode == 0) {
    // few parents: a block per child digit, so that the eight translations
    // of a chunk run side by side (64 parents at order 30: 0.37 ms in one
    // block each)
    const int nsplit = wide_m2m_nsplit(nb);
    const size_t C = (size_t)(Nout + 1) * (Nout + 1);
    double *part = nullptr;
    if (nsplit > 1 && dmalloc((void **)&part, sizeof(double) * 2 * nsplit * npar * C))
      return WBFMM_HIP_ERR_NOMEM;
    const int rc = launch_wide<0>("hel_m2m", dim3(nb, nsplit), parents, npar, ca, cstart, cend,
                                  nullptr, nullptr, 0, Nin, Nout, in, out, plan_dev, A, A2, CS,
                                  nsplit, part, npar, plan_host);
    if (!rc && nsplit > 1)
      WBFMM_LAUNCH("m2l_reduce", k_wide_m2m_sum, dim3((unsigned)((npar * C + 255) / 256)),
                   dim3(256), 0, parents, npar, (int)C, (const double2 *)part, (double2 *)out);
    dfree(part);
    return rc;
  }
  return launch_wide<1>("hel_l2l", dim3(nb, 8), parents, npar, ca, nullptr, nullptr, cflag,
                        nullptr, 0, Nin, Nout, in, out, plan_dev, A, A2, CS, 1, nullptr, npar,
                        plan_host);
}

}  // extern "C"
