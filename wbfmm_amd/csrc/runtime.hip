// runtime.hip -- stream, memory and timing services of the thin C ABI,
// plus the octree build kernels (Morton codes, stable sort, box ranges).
//
// Tree build restates src/boxes.c:118-277: the reference sorts an index
// array by Morton code with a stable qsort and then segments it level by
// level; here the codes are computed by one kernel, sorted with rocPRIM's
// stable LSD radix sort, and every level's [start,end) ranges are found by
// one kernel that marks segment boundaries in the sorted codes.

#include <cstdio>
#include <cstring>

#include <hip/hip_runtime.h>
#include <rocprim/rocprim.hpp>

#include <algorithm>
#include <map>
#include <mutex>
#include <string>
#include <unordered_map>
#include <vector>

#include "hip_common.h"

namespace wbfmm {

// The library stream, created by wbfmm_hip_init.  A thread may select
// another stream of its own (wbfmm_hip_set_stream); every launch, copy and
// stream-ordered allocation of that thread then goes there, which is how
// the serving engine runs independent solves side by side.
static hipStream_t g_stream = nullptr;
static thread_local hipStream_t t_stream = nullptr;
static std::mutex g_mu;
static thread_local char g_err[512] = "";
static bool g_timing = false;
static std::mutex g_timing_mu;
struct Ev {
  std::string name;
  hipEvent_t a, b;
};
static std::vector<Ev> g_events;
static std::map<std::string, std::pair<int, double>> g_totals;

hipStream_t stream() {
  if (t_stream) return t_stream;
  if (!g_stream) wbfmm_hip_init();
  return g_stream;
}

int fail(const char *what, hipError_t e) {
  snprintf(g_err, sizeof(g_err), "%s: %s", what, hipGetErrorString(e));
  fprintf(stderr, "wbfmm (HIP): %s\n", g_err);
  return WBFMM_HIP_ERR_RUNTIME;
}

int fail_msg(const char *msg, int code) {
  snprintf(g_err, sizeof(g_err), "%s", msg);
  fprintf(stderr, "wbfmm (HIP): %s\n", g_err);
  return code;
}

// Timing covers launches made on the library stream only; launches on a
// thread's own stream are not timed.
void timing_begin(const char *name) {
  if (!g_timing || t_stream) return;
  std::lock_guard<std::mutex> lk(g_timing_mu);
  Ev ev;
  ev.name = name;
  hipEventCreate(&ev.a);
  hipEventCreate(&ev.b);
  hipEventRecord(ev.a, g_stream);
  g_events.push_back(ev);
}

void timing_end(const char *name) {
  if (!g_timing || t_stream) return;
  (void)name;
  std::lock_guard<std::mutex> lk(g_timing_mu);
  hipEventRecord(g_events.back().b, g_stream);
}

static void timing_collect() {
  std::lock_guard<std::mutex> lk(g_timing_mu);
  if (g_events.empty()) return;
  hipStreamSynchronize(g_stream);
  for (auto &ev : g_events) {
    float ms = 0.0f;
    hipEventElapsedTime(&ms, ev.a, ev.b);
    auto &t = g_totals[ev.name];
    t.first += 1;
    t.second += ms;
    hipEventDestroy(ev.a);
    hipEventDestroy(ev.b);
  }
  g_events.clear();
}

// ---------------------------------------------------------------------
// tree kernels
// ---------------------------------------------------------------------

__global__ void k_morton(const char *pts, size_t pstr, unsigned n, double x0,
                         double y0, double z0, double D, double *xyz,
                         uint64_t *codes, uint32_t *idx, unsigned *nbad) {
  unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double *x = (const double *)(pts + (size_t)i * pstr);
  double a = x[0], b = x[1], c = x[2];
  if (a <= x0 || a >= x0 + D || b <= y0 || b >= y0 + D || c <= z0 ||
      c >= z0 + D)
    atomicAdd(nbad, 1u);
  codes[i] = point_code(a, b, c, x0, y0, z0, D);
  idx[i] = i;
  xyz[4 * (size_t)i + 0] = a;
  xyz[4 * (size_t)i + 1] = b;
  xyz[4 * (size_t)i + 2] = c;
  xyz[4 * (size_t)i + 3] = 0.0;
}

__global__ void k_stage4(const char *pts, size_t pstr, unsigned n,
                         double *out) {
  unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double *x = (const double *)(pts + (size_t)i * pstr);
  out[4 * (size_t)i + 0] = x[0];
  out[4 * (size_t)i + 1] = x[1];
  out[4 * (size_t)i + 2] = x[2];
  out[4 * (size_t)i + 3] = 0.0;
}

__global__ void k_gather4(const double *in, const uint32_t *idx, unsigned n,
                          double *out) {
  unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double *s = in + 4 * (size_t)idx[i];
  double *d = out + 4 * (size_t)i;
  d[0] = s[0];
  d[1] = s[1];
  d[2] = s[2];
  d[3] = s[3];
}

// Zero rows list[0..n) of planes of `rows' rows of rw words W: one wavefront
// per row, one plane per grid row; bound by the writes.  A solve of 1e6
// points on a sphere at depth 7 (5 % of its 2097152 leaf boxes of 4608 bytes
// hold points) spent 5.2 ms on fills of whole levels and now takes 46.3
// instead of 51.7 ms.
template <typename W>
__global__ __launch_bounds__(256) void k_clear_rows(W *p, const uint32_t *list, unsigned n,
                                                    size_t rows, unsigned rw) {
  const unsigned i = blockIdx.x * 4 + threadIdx.x / 64;
  if (i >= n) return;
  W *row = p + ((size_t)blockIdx.y * rows + list[i]) * rw;
  const W zero = {};
  for (unsigned w = threadIdx.x % 64; w < rw; w += 64) row[w] = zero;
}

// out record i = in record idx[i], records of rsize bytes moved as
// 4-byte words when rsize allows, else bytes
__global__ void k_gather_records4(const uint32_t *in, size_t rw, const uint32_t *idx,
                                  unsigned n, uint32_t *out) {
  const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (size_t)n * rw) return;
  const size_t i = e / rw, w = e % rw;
  out[e] = in[(size_t)idx[i] * rw + w];
}

__global__ void k_gather_records1(const uint8_t *in, size_t rsize, const uint32_t *idx,
                                  unsigned n, uint8_t *out) {
  const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (size_t)n * rsize) return;
  const size_t i = e / rsize, w = e % rsize;
  out[e] = in[(size_t)idx[i] * rsize + w];
}

__global__ void k_gather_strided(const double *src, int sstr, int ncomp,
                                 const uint32_t *idx, unsigned n,
                                 double *out) {
  unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  for (int c = 0; c < ncomp; c++)
    out[(size_t)i * ncomp + c] = src[(size_t)idx[i] * sstr + c];
}

__global__ void k_box_ranges(const uint64_t *codes, unsigned n, int shift,
                             uint32_t *start, uint32_t *end) {
  unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint64_t b = codes[i] >> shift;
  if (i == 0 || (codes[i - 1] >> shift) != b) start[b] = i;
  if (i == n - 1 || (codes[i + 1] >> shift) != b) end[b] = i + 1;
}

__global__ void k_box_flags(const uint32_t *start, const uint32_t *end,
                            unsigned nb, uint32_t *out) {
  unsigned b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nb) return;
  out[b] = end[b] > start[b];
}

__global__ void k_box_scatter(const uint32_t *flags, const uint32_t *pos,
                              unsigned nb, uint32_t *list) {
  unsigned b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nb) return;
  if (flags[b]) list[pos[b]] = b;
}

// ---- box ranges and box lists of all levels of a tree at once ----------------
//
// The boxes of the levels lo..lo+n-1 form one grid of 2048-box chunks.  Three
// launches, whatever the depth: the ranges (or flags) of every box with the
// chunk's counts; an exclusive scan of the counts over each level's chunks,
// one block a level, whose totals go to tot; the lists, each box placed by
// its chunk's base and its rank in the chunk.  Counts stay on the device and
// reach the host in one copy.  Level by level, with a library scan over a
// flag array and the count read back at each level, a tree of depth 2 took
// some 60 launches and copies and 7 waits for the device, twice over with a
// target list.
constexpr unsigned kLevChunk = 2048, kLevThreads = 256;
constexpr int kLevMax = 17;
struct LevelSet {
  unsigned lo, n;
  unsigned chunk0[kLevMax + 1];
  uint32_t *start[kLevMax], *end[kLevMax];                 // ranges over the sources
  uint32_t *list[kLevMax], *flag[kLevMax], *cls[kLevMax];  // lists; flags and class lists of targets
};

// first i with codes[i] >= key
__device__ __forceinline__ unsigned code_bound(const uint64_t *__restrict__ codes, unsigned n,
                                               uint64_t key) {
  unsigned a = 0, b = n;
  while (a < b) {
    const unsigned m = a + (b - a) / 2;
    if (codes[m] < key)
      a = m + 1;
    else
      b = m;
  }
  return a;
}

// level index (from lo) of the block's chunk, its first box and the number
// of boxes of the level
__device__ __forceinline__ int chunk_level(const LevelSet &L, unsigned &box0, unsigned &nb) {
  int l = 0;
  while (l + 1 < (int)L.n && blockIdx.x >= L.chunk0[l + 1]) l++;
  box0 = (blockIdx.x - L.chunk0[l]) * kLevChunk;
  nb = 1u << (3 * (L.lo + l));
  return l;
}

// [start, end) of every box over the sorted codes (0, 0 for an empty box)
__global__ __launch_bounds__(kLevThreads) void k_level_ranges(const uint64_t *__restrict__ codes,
                                                              unsigned n, LevelSet L,
                                                              uint32_t *__restrict__ cnt) {
  __shared__ unsigned bound[kLevThreads + 1], total;
  unsigned box0, nb;
  const int l = chunk_level(L, box0, nb), shift = 3 * (20 - (int)(L.lo + l));
  if (threadIdx.x == 0) total = 0;
  for (unsigned i = 0; i < kLevChunk; i += kLevThreads) {
    const unsigned b = box0 + i + threadIdx.x;
    __syncthreads();
    if (b < nb) {
      bound[threadIdx.x] = code_bound(codes, n, (uint64_t)b << shift);
      if (threadIdx.x == kLevThreads - 1 || b == nb - 1)
        bound[threadIdx.x + 1] = code_bound(codes, n, ((uint64_t)b + 1) << shift);
    }
    __syncthreads();
    bool occ = false;
    if (b < nb) {
      const unsigned s = bound[threadIdx.x], e = bound[threadIdx.x + 1];
      occ = e > s;
      L.start[l][b] = occ ? s : 0u;
      L.end[l][b] = occ ? e : 0u;
    }
    const unsigned c = (unsigned)__popcll(__ballot(occ));
    if ((threadIdx.x & 63) == 0 && c) atomicAdd(&total, c);
  }
  __syncthreads();
  if (threadIdx.x == 0) cnt[blockIdx.x] = total;
}

// flag of every box: 1 where it holds sources or targets; counts of the
// flagged boxes and of those of each child digit (9 per chunk)
__global__ __launch_bounds__(kLevThreads) void k_level_flags(const uint64_t *__restrict__ tcodes,
                                                             unsigned n, LevelSet L,
                                                             uint32_t *__restrict__ cnt) {
  __shared__ unsigned total[9];
  unsigned box0, nb;
  const int l = chunk_level(L, box0, nb), shift = 3 * (20 - (int)(L.lo + l));
  if (threadIdx.x < 9) total[threadIdx.x] = 0;
  __syncthreads();
  for (unsigned i = 0; i < kLevChunk; i += kLevThreads) {
    const unsigned b = box0 + i + threadIdx.x;
    bool on = false;
    if (b < nb) {
      on = L.end[l][b] > L.start[l][b];
      if (!on) {
        const unsigned s = code_bound(tcodes, n, (uint64_t)b << shift);
        on = s < n && (tcodes[s] >> shift) == b;
      }
      L.flag[l][b] = on ? 1u : 0u;
    }
    const unsigned long long m = __ballot(on);
    const int lane = threadIdx.x & 63;
    if (lane < 9 && m) {
      const unsigned c = (unsigned)__popcll(lane ? m & (0x0101010101010101ull << (lane - 1)) : m);
      if (c) atomicAdd(&total[lane], c);
    }
  }
  __syncthreads();
  if (threadIdx.x < 9) cnt[9 * (size_t)blockIdx.x + threadIdx.x] = total[threadIdx.x];
}

// counts of F fields per chunk -> exclusive sums over the chunks of the
// level; totals to tot[10 level + at + field] (block: a level)
template <int F>
__global__ __launch_bounds__(1024) void k_chunk_scan(LevelSet L, uint32_t *__restrict__ cnt,
                                                     uint32_t *__restrict__ tot, int at) {
  __shared__ unsigned wsum[16];
  const int l = blockIdx.x, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const unsigned c0 = L.chunk0[l], c1 = L.chunk0[l + 1];
  for (int f = 0; f < F; f++) {
    unsigned base = 0;
    for (unsigned c = c0; c < c1; c += 1024) {
      const unsigned k = c + threadIdx.x;
      const unsigned v = k < c1 ? cnt[(size_t)k * F + f] : 0u;
      unsigned x = v;
      for (int h = 1; h < 64; h *= 2) {
        const unsigned y = __shfl_up(x, h);
        if (lane >= h) x += y;
      }
      if (lane == 63) wsum[w] = x;
      __syncthreads();
      unsigned before = base, all = 0;
      for (int i = 0; i < 16; i++) {
        if (i < w) before += wsum[i];
        all += wsum[i];
      }
      if (k < c1) cnt[(size_t)k * F + f] = before + x - v;
      base += all;
      __syncthreads();
    }
    if (threadIdx.x == 0) tot[10 * (L.lo + l) + at + f] = base;
  }
}

// boxes in ascending order where end > start (CLS 0), or the flagged boxes
// in ascending order and grouped by child digit (CLS 1)
template <int CLS>
__global__ __launch_bounds__(kLevThreads) void k_level_lists(LevelSet L,
                                                             const uint32_t *__restrict__ base,
                                                             const uint32_t *__restrict__ tot) {
  constexpr int F = CLS ? 9 : 1, W = kLevThreads / 64;
  __shared__ unsigned wc[W][F];
  unsigned box0, nb;
  const int l = chunk_level(L, box0, nb), lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const unsigned digit = threadIdx.x & 7;
  const unsigned long long below = (1ull << lane) - 1, mine = 0x0101010101010101ull << digit;
  unsigned at = base[(size_t)blockIdx.x * F], cat = 0;
  if (CLS) {
    cat = base[(size_t)blockIdx.x * F + 1 + digit];
    for (unsigned c = 0; c < digit; c++) cat += tot[10 * (L.lo + l) + 2 + c];
  }
  for (unsigned i = 0; i < kLevChunk; i += kLevThreads) {
    const unsigned b = box0 + i + threadIdx.x;
    bool on = false;
    if (b < nb) on = CLS ? L.flag[l][b] != 0 : L.end[l][b] > L.start[l][b];
    const unsigned long long m = __ballot(on);
    __syncthreads();
    if (lane < F)
      wc[w][lane] = (unsigned)__popcll(lane ? m & (0x0101010101010101ull << (lane - 1)) : m);
    __syncthreads();
    unsigned r = (unsigned)__popcll(m & below), cr = (unsigned)__popcll(m & below & mine);
    for (int j = 0; j < W; j++) {
      if (j < w) {
        r += wc[j][0];
        if (CLS) cr += wc[j][F > 1 ? 1 + digit : 0];
      }
    }
    if (on) {
      L.list[l][at + r] = b;
      if (CLS) L.cls[l][cat + cr] = b;
    }
    for (int j = 0; j < W; j++) {
      at += wc[j][0];
      if (CLS) cat += wc[j][F > 1 ? 1 + digit : 0];
    }
  }
}

// every box of a level, grouped by child digit
__global__ void k_all_classes(unsigned nb, uint32_t *out) {
  const unsigned i = blockIdx.x * blockDim.x + threadIdx.x, per = nb / 8;
  if (i < nb) out[i] = 8 * (i % per) + i / per;
}

// per-block minimum and maximum of the 3 coordinates: out[6 b + 0..2] min,
// out[6 b + 3..5] max
__global__ void k_bounds(const char *pts, size_t pstr, unsigned n,
                         double *out) {
  __shared__ double red[6][256];
  double lo[3] = {INFINITY, INFINITY, INFINITY};
  double hi[3] = {-INFINITY, -INFINITY, -INFINITY};
  for (unsigned i = blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += gridDim.x * blockDim.x) {
    const double *x = (const double *)(pts + (size_t)i * pstr);
    for (int c = 0; c < 3; c++) {
      lo[c] = fmin(lo[c], x[c]);
      hi[c] = fmax(hi[c], x[c]);
    }
  }
  for (int c = 0; c < 3; c++) {
    red[c][threadIdx.x] = lo[c];
    red[3 + c][threadIdx.x] = hi[c];
  }
  __syncthreads();
  for (unsigned h = blockDim.x / 2; h > 0; h >>= 1) {
    if (threadIdx.x < h)
      for (int c = 0; c < 3; c++) {
        red[c][threadIdx.x] = fmin(red[c][threadIdx.x], red[c][threadIdx.x + h]);
        red[3 + c][threadIdx.x] =
            fmax(red[3 + c][threadIdx.x], red[3 + c][threadIdx.x + h]);
      }
    __syncthreads();
  }
  if (threadIdx.x < 6) out[6 * blockIdx.x + threadIdx.x] = red[threadIdx.x][0];
}

__global__ void k_accumulate(double *dst, int dstr, const double *src,
                             int sstr, int ncomp, unsigned n) {
  unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  for (int c = 0; c < ncomp; c++)
    dst[(size_t)i * dstr + c] += src[(size_t)i * sstr + c];
}

static inline unsigned nblk(size_t n, unsigned b) {
  return (unsigned)((n + b - 1) / b);
}


// allocations of this thread still to be refused, and calls of the runtime's
// allocator still to be answered as out of memory (failure-handling tests)
static thread_local int t_fail_allocs = 0, t_fail_mallocs = 0;

// Freed blocks kept for the next allocation on the same stream.  hipMallocAsync
// and hipFreeAsync take 10 to 70 us of host time each (the free of a block
// that queued work still uses most), and a solve of a small problem makes
// about twenty pairs: 1000 points 0.67 -> 0.49 ms, 20011 points 0.87 -> 0.72,
// 16 served problems 30 -> 16.
// A block freed on a stream is handed out on that stream only, where its next
// use is queued behind its last, as with hipFreeAsync; streams that the library
// did not create, whose end it does not see, and streams under capture, whose
// blocks belong to the graph, take the runtime's allocator.  At most 1 GiB is
// kept, in blocks up to 256 MiB (a level array of a large tree is worth a
// call) and at most 16384 of them, the longest unused given back first; a
// stream's blocks are given back before it is destroyed, and every stream's
// when the runtime has no memory for an allocation, of any size and on any
// stream that is not under capture (pool_give_back), which is then tried once
// more.  Blocks of a stream that is being captured stay until the capture has
// ended.  An allocation looks through its own stream's blocks: with its free
// 0.8 us when few are kept, 4.3 with 16384.  10 served problems of 1000 to
// 12300 points take 2.70 ms; 2.84 with one list for all streams, 3.02 with
// ordered maps, whose nodes several threads allocate and free under the lock.
constexpr size_t kPoolBytes = (size_t)1 << 30, kPoolBlock = (size_t)256 << 20, kPoolCount = 16384;
struct PoolBlock {
  void *p;
  size_t bytes;
  uint64_t stamp;
};
struct PoolStream {
  hipStream_t s;
  std::vector<PoolBlock> free;
};
// (never destroyed: blocks may be freed while the process ends)
static std::mutex &g_pool_mu = *new std::mutex;
static auto &g_pool = *new std::vector<PoolStream>;  // the library's own streams
static auto &g_pool_live = *new std::unordered_map<void *, size_t>;  // blocks handed out
static size_t g_pool_bytes = 0, g_pool_count = 0;  // kept, of all streams
static uint64_t g_pool_stamp = 0;

// b becomes the size of block p, handed out; false when the host has no
// memory for the entry.  An entry may be there: of a block that its holder
// gave to hipFree, whose address has come back with another size.
static bool pool_note(void *p, size_t b) {
  try {
    g_pool_live[p] = b;
    return true;
  } catch (...) {
    return false;
  }
}

static bool capturing(hipStream_t s) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  return hipStreamIsCapturing(s, &st) != hipSuccess || st != hipStreamCaptureStatusNone;
}

// the kept blocks of stream s, null for streams that are not the library's
// own (g_pool_mu held)
static PoolStream *pool_of(hipStream_t s) {
  for (PoolStream &q : g_pool)
    if (q.s == s) return &q;
  return nullptr;
}

static void pool_add_stream(hipStream_t s) {
  std::lock_guard<std::mutex> lk(g_pool_mu);
  try {
    g_pool.push_back(PoolStream{s, {}});
  } catch (...) {  // a stream that is not listed takes the runtime's allocator
  }
}

// take free block i out of the list (g_pool_mu held)
static PoolBlock pool_take(PoolStream &q, size_t i) {
  const PoolBlock b = q.free[i];
  q.free[i] = q.free.back();
  q.free.pop_back();
  g_pool_bytes -= b.bytes;
  g_pool_count--;
  return b;
}

// give free block i back to the runtime (g_pool_mu held); false, and the block
// stays, while its stream is under capture (the free would be refused or
// become part of that graph)
static bool pool_release(PoolStream &q, size_t i) {
  if (capturing(q.s)) return false;
  if (hipFreeAsync(q.free[i].p, q.s) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  (void)pool_take(q, i);
  return true;
}

// give back the free blocks of stream s, or of all streams (null)
static void pool_flush(hipStream_t s) {
  std::lock_guard<std::mutex> lk(g_pool_mu);
  for (PoolStream &q : g_pool)
    for (size_t i = !s || q.s == s ? q.free.size() : 0; i-- > 0;) (void)pool_release(q, i);
}

// release free blocks, the longest unused first, until `bytes' more may be
// kept (g_pool_mu held); false when those that are left cannot be released
static bool pool_make_room(size_t bytes) {
  while (g_pool_bytes + bytes > kPoolBytes || g_pool_count >= kPoolCount) {
    PoolStream *of = nullptr;
    size_t old = 0;
    for (PoolStream &q : g_pool) {
      if (q.free.empty() || capturing(q.s)) continue;
      for (size_t i = 0; i < q.free.size(); i++)
        if (!of || q.free[i].stamp < of->free[old].stamp) {
          of = &q;
          old = i;
        }
    }
    if (!of || !pool_release(*of, old)) return false;
  }
  return true;
}

// give every free block back, wait until its stream is done with it, and
// let the runtime return what it holds unused to the device: the memory may
// be wanted on another stream or in a larger piece.  False when none was
// released.  The lock is held throughout, so that no stream of a block ends
// here.
static bool pool_give_back() {
  std::lock_guard<std::mutex> lk(g_pool_mu);
  std::vector<hipStream_t> used;
  try {
    used.reserve(g_pool.size());
  } catch (...) {  // no host memory either
    return false;
  }
  for (PoolStream &q : g_pool) {
    const size_t had = q.free.size();
    for (size_t i = had; i-- > 0;) (void)pool_release(q, i);
    if (q.free.size() < had) used.push_back(q.s);
  }
  if (used.empty()) return false;
  for (hipStream_t s : used) (void)hipStreamSynchronize(s);
  int dev = 0;
  hipMemPool_t pool;
  if (hipGetDevice(&dev) == hipSuccess && hipDeviceGetDefaultMemPool(&pool, dev) == hipSuccess)
    (void)hipMemPoolTrimTo(pool, 0);
  return true;
}

static hipError_t runtime_malloc(void **p, size_t bytes, hipStream_t s) {
  if (t_fail_mallocs > 0) {
    t_fail_mallocs--;
    return hipErrorOutOfMemory;
  }
  return hipMallocAsync(p, bytes, s);
}

int dmalloc(void **p, size_t bytes) {
  *p = nullptr;
  if (t_fail_allocs > 0) {
    t_fail_allocs--;
    return fail_msg("device allocation refused (forced by wbfmm_hip_debug_fail_allocs)",
                    WBFMM_HIP_ERR_NOMEM);
  }
  if (bytes == 0) bytes = 256;
  const hipStream_t s = stream();
  bool pooled = false;
  if (bytes <= kPoolBlock && !capturing(s)) {
    std::lock_guard<std::mutex> lk(g_pool_mu);
    if (PoolStream *q = pool_of(s)) {
      pooled = true;
      const size_t most = bytes + bytes / 4 + 4096, n = q->free.size();
      size_t best = n;
      // the smallest that fits, no more than a quarter (or a page) too large
      for (size_t i = 0; i < n; i++) {
        const size_t b = q->free[i].bytes;
        if (b >= bytes && b <= most && (best == n || b < q->free[best].bytes)) best = i;
      }
      if (best < n && pool_note(q->free[best].p, q->free[best].bytes)) {
        *p = pool_take(*q, best).p;
        return 0;
      }
    }
  }
  hipError_t e = runtime_malloc(p, bytes, s);
  if (e != hipSuccess && !capturing(s)) {
    (void)hipGetLastError();
    if (pool_give_back()) e = runtime_malloc(p, bytes, s);
  }
  if (e != hipSuccess) {
    *p = nullptr;
    fail("hipMallocAsync", e);
    return WBFMM_HIP_ERR_NOMEM;
  }
  {
    std::lock_guard<std::mutex> lk(g_pool_mu);
    if (!pooled || !pool_note(*p, bytes)) g_pool_live.erase(*p);
  }
  return 0;
}

static hipError_t free_block(void *p) {
  const hipStream_t s = stream();
  const bool keep = !capturing(s);
  {
    std::lock_guard<std::mutex> lk(g_pool_mu);
    const auto it = g_pool_live.find(p);
    if (it != g_pool_live.end()) {
      const size_t bytes = it->second;
      g_pool_live.erase(it);
      PoolStream *q = keep ? pool_of(s) : nullptr;
      if (q && pool_make_room(bytes)) {
        try {
          q->free.push_back(PoolBlock{p, bytes, g_pool_stamp++});
          g_pool_bytes += bytes;
          g_pool_count++;
          return hipSuccess;
        } catch (...) {  // no host memory for the entry: to the runtime
        }
      }
    }
  }
  return hipFreeAsync(p, s);
}

void dfree(void *p) {
  if (p) (void)free_block(p);
}

}  // namespace wbfmm

using namespace wbfmm;

extern "C" {

int wbfmm_hip_init(void) {
  std::lock_guard<std::mutex> lk(g_mu);
  if (g_stream) return 0;
  int ndev = 0;
  hipError_t e = hipGetDeviceCount(&ndev);
  if (e != hipSuccess || ndev < 1) {
    snprintf(g_err, sizeof(g_err), "no HIP device available (%s)",
             hipGetErrorString(e));
    fprintf(stderr, "wbfmm (HIP): %s\n", g_err);
    return WBFMM_HIP_ERR_RUNTIME;
  }
  // freed blocks stay in the default pool instead of going back to the
  // driver, so the per-solve allocations are served from the pool
  int dev = 0;
  WBFMM_CHECK(hipGetDevice(&dev));
  hipMemPool_t pool;
  WBFMM_CHECK(hipDeviceGetDefaultMemPool(&pool, dev));
  uint64_t keep = UINT64_MAX;
  WBFMM_CHECK(hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &keep));
  // default priority, non-blocking with respect to the null stream
  hipStream_t h = nullptr;
  WBFMM_CHECK(hipStreamCreateWithFlags(&h, hipStreamNonBlocking));
  pool_add_stream(h);
  g_stream = h;
  return 0;
}

int wbfmm_hip_mem_info(size_t *free_bytes, size_t *total_bytes) {
  if (wbfmm_hip_init()) return WBFMM_HIP_ERR_RUNTIME;
  WBFMM_CHECK(hipMemGetInfo(free_bytes, total_bytes));
  return 0;
}

int wbfmm_hip_stream_create(void **s) {
  if (wbfmm_hip_init()) return WBFMM_HIP_ERR_RUNTIME;
  hipStream_t h = nullptr;
  WBFMM_CHECK(hipStreamCreateWithFlags(&h, hipStreamNonBlocking));
  pool_add_stream(h);
  *s = (void *)h;
  return 0;
}

int wbfmm_hip_stream_destroy(void *s) {
  if (!s) return 0;
  WBFMM_CHECK(hipStreamSynchronize((hipStream_t)s));
  pool_flush((hipStream_t)s);
  {
    std::lock_guard<std::mutex> lk(g_pool_mu);
    for (size_t i = 0; i < g_pool.size(); i++)
      if (g_pool[i].s == (hipStream_t)s) {
        while (!g_pool[i].free.empty()) (void)pool_take(g_pool[i], 0);  // (refused by the runtime)
        g_pool.erase(g_pool.begin() + (ptrdiff_t)i);
        break;
      }
  }
  WBFMM_CHECK(hipStreamSynchronize((hipStream_t)s));
  WBFMM_CHECK(hipStreamDestroy((hipStream_t)s));
  return 0;
}

static thread_local int t_variant[WBFMM_VARIANT_COUNT] = {-1, -1};

int wbfmm_hip_set_variant(int which, int value) {
  // M2L: -1..2; field: -1..1
  const int vmax = which == WBFMM_VARIANT_FIELD ? 1 : 2;
  if (which < 0 || which >= WBFMM_VARIANT_COUNT || value < -1 || value > vmax)
    return fail_msg("unknown kernel variant", WBFMM_HIP_ERR_ARG);
  t_variant[which] = value;
  return 0;
}

int wbfmm_hip_get_variant(int which) {
  return which >= 0 && which < WBFMM_VARIANT_COUNT ? t_variant[which] : -1;
}

int wbfmm_hip_set_stream(void *s, void **prev) {
  if (prev) *prev = (void *)t_stream;
  t_stream = (hipStream_t)s;
  return 0;
}

void *wbfmm_hip_get_stream(void) { return (void *)stream(); }

const char *wbfmm_hip_last_error(void) { return g_err; }

int wbfmm_hip_debug_fail_allocs(int n) {
  t_fail_allocs = n > 0 ? n : 0;
  return 0;
}

int wbfmm_hip_debug_fail_mallocs(int n) {
  t_fail_mallocs = n > 0 ? n : 0;
  return 0;
}

int wbfmm_hip_malloc(void **p, size_t bytes) {
  if (wbfmm_hip_init()) return WBFMM_HIP_ERR_RUNTIME;
  return dmalloc(p, bytes);
}

int wbfmm_hip_free(void *p) {
  if (!p) return 0;
  WBFMM_CHECK(free_block(p));
  return 0;
}

size_t wbfmm_hip_pool_bytes(void) {
  std::lock_guard<std::mutex> lk(g_pool_mu);
  return g_pool_bytes;
}

int wbfmm_hip_pool_release(void) {
  pool_flush(nullptr);
  return 0;
}

int wbfmm_hip_is_device(const void *p) {
  if (!p) return 0;
  if (wbfmm_hip_init()) return 0;
  hipPointerAttribute_t a;
  hipError_t e = hipPointerGetAttributes(&a, p);
  if (e != hipSuccess) {
    hipGetLastError();  // clear the sticky error from an unknown pointer
    return 0;
  }
  return a.type == hipMemoryTypeDevice || a.type == hipMemoryTypeManaged;
}

int wbfmm_hip_memcpy(void *dst, const void *src, size_t bytes) {
  if (bytes == 0) return 0;
  WBFMM_CHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDefault, stream()));
  if (!wbfmm_hip_is_device(dst) || !wbfmm_hip_is_device(src))
    WBFMM_CHECK(hipStreamSynchronize(stream()));
  return 0;
}

int wbfmm_hip_memset(void *p, int v, size_t bytes) {
  if (bytes == 0) return 0;
  WBFMM_CHECK(hipMemsetAsync(p, v, bytes, stream()));
  return 0;
}

int wbfmm_hip_sync(void) {
  WBFMM_CHECK(hipStreamSynchronize(stream()));
  return 0;
}

int wbfmm_hip_timing_enable(int on) {
  timing_collect();
  g_timing = (on != 0);
  return 0;
}

int wbfmm_hip_timing_reset(void) {
  timing_collect();
  g_totals.clear();
  return 0;
}

int wbfmm_hip_timing_query(const char *name, int *launches, double *ms) {
  timing_collect();
  auto it = g_totals.find(name);
  if (it == g_totals.end()) {
    *launches = 0;
    *ms = 0.0;
    return 0;
  }
  *launches = it->second.first;
  *ms = it->second.second;
  return 0;
}

int wbfmm_hip_morton(const void *pts, size_t pstr, unsigned n,
                     const double *x0, double D, double *xyz,
                     uint64_t *codes, uint32_t *idx, unsigned *nbad) {
  if (n == 0) {
    *nbad = 0;
    return 0;
  }
  const char *dpts = (const char *)pts;
  void *staged = nullptr;
  if (!wbfmm_hip_is_device(pts)) {
    // copy the strided host block as it lies
    size_t bytes = (size_t)(n - 1) * pstr + 3 * sizeof(double);
    if (wbfmm_hip_malloc(&staged, bytes)) return WBFMM_HIP_ERR_NOMEM;
    WBFMM_CHECK(hipMemcpyAsync(staged, pts, bytes, hipMemcpyHostToDevice,
                               stream()));
    dpts = (const char *)staged;
  }
  unsigned *dbad = nullptr;
  if (dmalloc((void **)&dbad, sizeof(unsigned))) return WBFMM_HIP_ERR_NOMEM;
  WBFMM_CHECK(hipMemsetAsync(dbad, 0, sizeof(unsigned), stream()));
  WBFMM_LAUNCH("tree_morton", k_morton, dim3(nblk(n, 256)), dim3(256), 0,
               dpts, pstr, n, x0[0], x0[1], x0[2], D, xyz, codes, idx, dbad);
  WBFMM_CHECK(hipMemcpyAsync(nbad, dbad, sizeof(unsigned),
                             hipMemcpyDeviceToHost, stream()));
  dfree(dbad);
  dfree(staged);
  WBFMM_CHECK(hipStreamSynchronize(stream()));
  return 0;
}

int wbfmm_hip_stage4(const void *pts, size_t pstr, unsigned n, double *out) {
  if (n == 0) return 0;
  const char *dpts = (const char *)pts;
  void *staged = nullptr;
  if (!wbfmm_hip_is_device(pts)) {
    size_t bytes = (size_t)(n - 1) * pstr + 3 * sizeof(double);
    if (wbfmm_hip_malloc(&staged, bytes)) return WBFMM_HIP_ERR_NOMEM;
    WBFMM_CHECK(hipMemcpyAsync(staged, pts, bytes, hipMemcpyHostToDevice,
                               stream()));
    dpts = (const char *)staged;
  }
  WBFMM_LAUNCH("stage4", k_stage4, dim3(nblk(n, 256)), dim3(256), 0, dpts,
               pstr, n, out);
  if (staged) {
    dfree(staged);
    // the caller's host block may be reused once this returns
    WBFMM_CHECK(hipStreamSynchronize(stream()));
  }
  return 0;
}

int wbfmm_hip_sort(uint64_t *codes, uint32_t *idx, unsigned n) {
  if (n < 2) return 0;
  uint64_t *k2 = nullptr;
  uint32_t *v2 = nullptr;
  void *tmp = nullptr;
  if (dmalloc((void **)&k2, sizeof(uint64_t) * n) ||
      dmalloc((void **)&v2, sizeof(uint32_t) * n))
    return WBFMM_HIP_ERR_NOMEM;
  size_t bytes = 0;
  WBFMM_CHECK(rocprim::radix_sort_pairs(nullptr, bytes, codes, k2, idx, v2,
                                        n, 0, 60, stream()));
  if (dmalloc(&tmp, bytes)) return WBFMM_HIP_ERR_NOMEM;
  timing_begin("tree_sort");
  WBFMM_CHECK(rocprim::radix_sort_pairs(tmp, bytes, codes, k2, idx, v2, n,
                                        0, 60, stream()));
  timing_end("tree_sort");
  WBFMM_CHECK(hipMemcpyAsync(codes, k2, sizeof(uint64_t) * n,
                             hipMemcpyDeviceToDevice, stream()));
  WBFMM_CHECK(hipMemcpyAsync(idx, v2, sizeof(uint32_t) * n,
                             hipMemcpyDeviceToDevice, stream()));
  dfree(tmp);
  dfree(k2);
  dfree(v2);
  return 0;
}

int wbfmm_hip_clear_rows(void *p, const uint32_t *list, unsigned n, size_t rows,
                         size_t row_bytes, unsigned planes) {
  if (n == 0 || planes == 0 || row_bytes == 0) return 0;
  if (row_bytes % 4 || (uintptr_t)p % 4 || planes > 65535 || row_bytes / 4 > 0xffffffffu)
    return WBFMM_HIP_ERR_ARG;
  const size_t a = (uintptr_t)p | row_bytes;  // the widest words that p and the rows allow
  const dim3 grid(nblk(n, 4), planes);
  if (a % 16 == 0)
    WBFMM_LAUNCH("clear_rows", (k_clear_rows<uint4>), grid, dim3(256), 0, (uint4 *)p, list, n,
                 rows, (unsigned)(row_bytes / 16));
  else if (a % 8 == 0)
    WBFMM_LAUNCH("clear_rows", (k_clear_rows<uint2>), grid, dim3(256), 0, (uint2 *)p, list, n,
                 rows, (unsigned)(row_bytes / 8));
  else
    WBFMM_LAUNCH("clear_rows", (k_clear_rows<uint32_t>), grid, dim3(256), 0, (uint32_t *)p, list,
                 n, rows, (unsigned)(row_bytes / 4));
  return 0;
}

int wbfmm_hip_gather4(const double *in, const uint32_t *idx, unsigned n,
                      double *out) {
  if (n == 0) return 0;
  WBFMM_LAUNCH("gather4", k_gather4, dim3(nblk(n, 256)), dim3(256), 0, in,
               idx, n, out);
  return 0;
}

int wbfmm_hip_gather_strided(const double *src, int sstr, int ncomp,
                             const uint32_t *idx, unsigned n, double *out) {
  if (n == 0) return 0;
  if (sstr < ncomp) return WBFMM_HIP_ERR_ARG;
  const double *dsrc = src;
  void *staged = nullptr;
  if (!wbfmm_hip_is_device(src)) {
    size_t bytes = sizeof(double) * ((size_t)(n - 1) * sstr + ncomp);
    // the index range covers 0..n-1 (a permutation of the input)
    if (wbfmm_hip_malloc(&staged, bytes)) return WBFMM_HIP_ERR_NOMEM;
    WBFMM_CHECK(hipMemcpyAsync(staged, src, bytes, hipMemcpyHostToDevice,
                               stream()));
    dsrc = (const double *)staged;
  }
  WBFMM_LAUNCH("gather_strength", k_gather_strided, dim3(nblk(n, 256)),
               dim3(256), 0, dsrc, sstr, ncomp, idx, n, out);
  if (staged) {
    dfree(staged);
    WBFMM_CHECK(hipStreamSynchronize(stream()));
  }
  return 0;
}

int wbfmm_hip_gather_records(const void *in, size_t rsize, const uint32_t *idx, unsigned n,
                             void *out) {
  if (n == 0) return 0;
  if (rsize == 0) return WBFMM_HIP_ERR_ARG;
  if (rsize % 4 == 0 && (uintptr_t)in % 4 == 0 && (uintptr_t)out % 4 == 0) {
    const size_t rw = rsize / 4, tot = (size_t)n * rw;
    WBFMM_LAUNCH("gather_records", k_gather_records4, dim3((unsigned)((tot + 255) / 256)),
                 dim3(256), 0, (const uint32_t *)in, rw, idx, n, (uint32_t *)out);
  } else {
    const size_t tot = (size_t)n * rsize;
    WBFMM_LAUNCH("gather_records", k_gather_records1, dim3((unsigned)((tot + 255) / 256)),
                 dim3(256), 0, (const uint8_t *)in, rsize, idx, n, (uint8_t *)out);
  }
  return 0;
}

int wbfmm_hip_box_ranges(const uint64_t *codes, unsigned n, unsigned level,
                         uint32_t *start, uint32_t *end) {
  size_t nb = (size_t)1 << (3 * level);
  WBFMM_CHECK(hipMemsetAsync(start, 0, sizeof(uint32_t) * nb, stream()));
  WBFMM_CHECK(hipMemsetAsync(end, 0, sizeof(uint32_t) * nb, stream()));
  if (n == 0) return 0;
  WBFMM_LAUNCH("tree_box_ranges", k_box_ranges, dim3(nblk(n, 256)),
               dim3(256), 0, codes, n, (int)(3 * (20 - level)), start, end);
  return 0;
}

int wbfmm_hip_compact_boxes(const uint32_t *start, const uint32_t *end,
                            unsigned level, uint32_t *list, unsigned *count) {
  unsigned nb = 1u << (3 * level);
  uint32_t *flags = nullptr, *pos = nullptr;
  void *tmp = nullptr;
  if (dmalloc((void **)&flags, sizeof(uint32_t) * nb) ||
      dmalloc((void **)&pos, sizeof(uint32_t) * nb))
    return WBFMM_HIP_ERR_NOMEM;
  WBFMM_LAUNCH("tree_box_flags", k_box_flags, dim3(nblk(nb, 256)), dim3(256),
               0, start, end, nb, flags);
  size_t bytes = 0;
  WBFMM_CHECK(rocprim::exclusive_scan(nullptr, bytes, flags, pos, 0u, nb,
                                      rocprim::plus<uint32_t>(), stream()));
  if (dmalloc(&tmp, bytes)) return WBFMM_HIP_ERR_NOMEM;
  WBFMM_CHECK(rocprim::exclusive_scan(tmp, bytes, flags, pos, 0u, nb,
                                      rocprim::plus<uint32_t>(), stream()));
  WBFMM_LAUNCH("tree_box_scatter", k_box_scatter, dim3(nblk(nb, 256)),
               dim3(256), 0, flags, pos, nb, list);
  uint32_t lastf = 0, lastp = 0;
  WBFMM_CHECK(hipMemcpyAsync(&lastf, flags + nb - 1, 4, hipMemcpyDeviceToHost,
                             stream()));
  WBFMM_CHECK(hipMemcpyAsync(&lastp, pos + nb - 1, 4, hipMemcpyDeviceToHost,
                             stream()));
  dfree(tmp);
  dfree(flags);
  dfree(pos);
  WBFMM_CHECK(hipStreamSynchronize(stream()));
  *count = lastf + lastp;
  return 0;
}

// points in Morton order: positions (4 doubles), codes and caller indices;
// raw: scratch of 4 n doubles; *nbad: points outside the domain; low: the
// lowest bits of the codes left out of the order (a multiple of 3: points
// of one box of level 20 - low / 3 keep the caller's order)
int wbfmm_hip_points_sorted(const void *pts, size_t pstr, unsigned n, const double *x0, double D,
                            int low, double *raw, double *xyz, uint64_t *codes, uint32_t *idx,
                            unsigned *nbad) {
  *nbad = 0;
  if (low < 0 || low > 57) return WBFMM_HIP_ERR_ARG;
  if (n == 0) return 0;
  size_t sort_bytes = 0;
  WBFMM_CHECK(rocprim::radix_sort_pairs(nullptr, sort_bytes, codes, codes, idx, idx, n, low, 60,
                                        stream()));
  // one block: counter, unsorted codes and indices, the caller's strided
  // host block as it lies, the sort's scratch
  const bool host = !wbfmm_hip_is_device(pts);
  auto round = [](size_t b) { return (b + 255) / 256 * 256; };
  const size_t o_codes = 256, o_idx = o_codes + round(8 * (size_t)n),
               o_pts = o_idx + round(4 * (size_t)n),
               pbytes = host ? (size_t)(n - 1) * pstr + 3 * sizeof(double) : 0,
               o_sort = o_pts + round(pbytes);
  char *tmp = nullptr;
  if (dmalloc((void **)&tmp, o_sort + sort_bytes)) return WBFMM_HIP_ERR_NOMEM;
  uint64_t *tcodes = (uint64_t *)(tmp + o_codes);
  uint32_t *tidx = (uint32_t *)(tmp + o_idx);
  const char *dpts = (const char *)pts;
  if (host) {
    WBFMM_CHECK(hipMemcpyAsync(tmp + o_pts, pts, pbytes, hipMemcpyHostToDevice, stream()));
    dpts = tmp + o_pts;
  }
  WBFMM_CHECK(hipMemsetAsync(tmp, 0, sizeof(unsigned), stream()));
  WBFMM_LAUNCH("tree_morton", k_morton, dim3(nblk(n, 256)), dim3(256), 0, dpts, pstr, n, x0[0],
               x0[1], x0[2], D, raw, tcodes, tidx, (unsigned *)tmp);
  timing_begin("tree_sort");
  WBFMM_CHECK(rocprim::radix_sort_pairs(tmp + o_sort, sort_bytes, tcodes, codes, tidx, idx, n,
                                        low, 60, stream()));
  timing_end("tree_sort");
  WBFMM_LAUNCH("gather4", k_gather4, dim3(nblk(n, 256)), dim3(256), 0, raw, idx, n, xyz);
  WBFMM_CHECK(hipMemcpyAsync(nbad, tmp, sizeof(unsigned), hipMemcpyDeviceToHost, stream()));
  dfree(tmp);
  WBFMM_CHECK(hipStreamSynchronize(stream()));
  return 0;
}

static int level_set(LevelSet &L, unsigned lo, unsigned hi, unsigned *chunks) {
  if (hi < lo || hi > (unsigned)kMortonAddMaxLevel) return WBFMM_HIP_ERR_ARG;
  L.lo = lo;
  L.n = hi - lo + 1;
  unsigned c = 0;
  for (unsigned i = 0; i < L.n; i++) {
    L.chunk0[i] = c;
    c += ((1u << (3 * (lo + i))) + kLevChunk - 1) / kLevChunk;
  }
  L.chunk0[L.n] = c;
  *chunks = c;
  return 0;
}

int wbfmm_hip_tree_levels(const uint64_t *codes, unsigned n, unsigned lo, unsigned hi,
                          uint32_t *const *start, uint32_t *const *end, uint32_t *const *occ,
                          uint32_t *tot) {
  LevelSet L{};
  unsigned chunks = 0;
  if (level_set(L, lo, hi, &chunks)) return WBFMM_HIP_ERR_ARG;
  for (unsigned i = 0; i < L.n; i++) {
    L.start[i] = start[lo + i];
    L.end[i] = end[lo + i];
    L.list[i] = occ[lo + i];
  }
  uint32_t *cnt = nullptr;
  if (dmalloc((void **)&cnt, sizeof(uint32_t) * chunks)) return WBFMM_HIP_ERR_NOMEM;
  WBFMM_LAUNCH("tree_box_ranges", k_level_ranges, dim3(chunks), dim3(kLevThreads), 0, codes, n, L,
               cnt);
  WBFMM_LAUNCH("tree_box_scan", k_chunk_scan<1>, dim3(L.n), dim3(1024), 0, L, cnt, tot, 0);
  WBFMM_LAUNCH("tree_box_lists", k_level_lists<0>, dim3(chunks), dim3(kLevThreads), 0, L, cnt, tot);
  dfree(cnt);
  return 0;
}

int wbfmm_hip_tree_targets(const uint64_t *tcodes, unsigned n, unsigned hi,
                           uint32_t *const *start, uint32_t *const *end, uint32_t *const *flag,
                           uint32_t *const *act, uint32_t *const *cls, uint32_t *tot) {
  LevelSet L{};
  unsigned chunks = 0;
  if (level_set(L, 0, hi, &chunks)) return WBFMM_HIP_ERR_ARG;
  for (unsigned i = 0; i < L.n; i++) {
    L.start[i] = start[i];
    L.end[i] = end[i];
    L.flag[i] = flag[i];
    L.list[i] = act[i];
    L.cls[i] = cls[i];
  }
  uint32_t *cnt = nullptr;
  if (dmalloc((void **)&cnt, sizeof(uint32_t) * 9 * chunks)) return WBFMM_HIP_ERR_NOMEM;
  WBFMM_LAUNCH("tree_box_flags", k_level_flags, dim3(chunks), dim3(kLevThreads), 0, tcodes, n, L,
               cnt);
  WBFMM_LAUNCH("tree_box_scan", k_chunk_scan<9>, dim3(L.n), dim3(1024), 0, L, cnt, tot, 1);
  WBFMM_LAUNCH("tree_box_lists", k_level_lists<1>, dim3(chunks), dim3(kLevThreads), 0, L, cnt, tot);
  dfree(cnt);
  return 0;
}

int wbfmm_hip_all_classes(unsigned level, uint32_t *out) {
  if (level < 1 || level > (unsigned)kMortonAddMaxLevel) return WBFMM_HIP_ERR_ARG;
  const unsigned nb = 1u << (3 * level);
  WBFMM_LAUNCH("tree_all_classes", k_all_classes, dim3(nblk(nb, 256)), dim3(256), 0, nb, out);
  return 0;
}

int wbfmm_hip_bounds(const void *pts, size_t pstr, unsigned n, double *lo,
                     double *hi) {
  for (int c = 0; c < 3; c++) {
    lo[c] = INFINITY;
    hi[c] = -INFINITY;
  }
  if (n == 0) return 0;
  if (!wbfmm_hip_is_device(pts)) {
    for (unsigned i = 0; i < n; i++) {
      const double *x = (const double *)((const char *)pts + (size_t)i * pstr);
      for (int c = 0; c < 3; c++) {
        lo[c] = fmin(lo[c], x[c]);
        hi[c] = fmax(hi[c], x[c]);
      }
    }
    return 0;
  }
  const unsigned nb = nblk(n, 256) < 512 ? nblk(n, 256) : 512;
  double *d = nullptr;
  if (dmalloc((void **)&d, sizeof(double) * 6 * nb)) return WBFMM_HIP_ERR_NOMEM;
  std::vector<double> h(6 * (size_t)nb);
  WBFMM_LAUNCH("bounds", k_bounds, dim3(nb), dim3(256), 0,
               (const char *)pts, pstr, n, d);
  WBFMM_CHECK(hipMemcpyAsync(h.data(), d, sizeof(double) * 6 * nb,
                             hipMemcpyDeviceToHost, stream()));
  dfree(d);
  WBFMM_CHECK(hipStreamSynchronize(stream()));
  for (unsigned b = 0; b < nb; b++)
    for (int c = 0; c < 3; c++) {
      lo[c] = fmin(lo[c], h[6 * b + c]);
      hi[c] = fmax(hi[c], h[6 * b + 3 + c]);
    }
  return 0;
}

int wbfmm_hip_accumulate(double *dst, int dstr, const double *src, int sstr,
                         int ncomp, unsigned n) {
  if (n == 0) return 0;
  if (dstr < ncomp || sstr < ncomp) return WBFMM_HIP_ERR_ARG;
  WBFMM_LAUNCH("accumulate", k_accumulate, dim3(nblk(n, 256)), dim3(256), 0,
               dst, dstr, src, sstr, ncomp, n);
  return 0;
}

}  // extern "C"
