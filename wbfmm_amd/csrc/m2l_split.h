// m2l_split.h -- how the M2L of a level with few targets is split over blocks,
// and what its partial sums take: one rule for the launches and for the
// serving engine's estimate of a solve's memory.  Plain C++, no HIP.
#pragma once

#include <cstddef>

namespace wbfmm {

// Blocks per chunk of the split M2L form (a chunk's offsets dealt to several
// blocks, whose partial sums k_m2l_reduce adds): levels with fewer than 1024
// chunks take up to 2048 blocks in all, at most 8 a chunk, and levels 2 and 3,
// where that leaves most of the chip idle while each block works through its
// offsets in series, up to 25.  With 8 there, level 2 (64 boxes) took 0.077 ms
// at order 8 and takes 0.035, levels 2 and 3 at order 13 0.217 and 0.152, 9
// launches of 3 components at order 10 1.52 and 1.40; 35 a chunk or 4096
// blocks gain nothing more, and their partial sums cost more.  More than 8
// only while a full level's partials stay within kSplitBytes, the memory of
// the allocation-free entry point.  The split depends on the level, the order
// and the chunk count alone, so that a problem always sums in the same order
// (up to 256 chunks, as a Laplace level 4 has, not on the count either).
constexpr size_t kSplitBytes = ((size_t)62 << 20) - ((size_t)16 << 10);
inline unsigned m2l_split_most(int level, size_t bytes_per_box) {
  if (level > 3) return 8;
  const size_t fit = kSplitBytes / (bytes_per_box << (3 * level));
  return fit < 8 ? 8 : fit < 25 ? (unsigned)fit : 25;
}
inline int m2l_nsplit(int level, unsigned nchunks, size_t bytes_per_box) {
  if (nchunks >= 1024) return 1;
  const unsigned most = m2l_split_most(level, bytes_per_box);
  return (int)(2048 / nchunks < most ? 2048 / nchunks : most);
}
// the expansions that a level's partial sums hold at most, whatever its
// targets: chunks of up to 16, so 2048 blocks hold no more than 32768
inline size_t m2l_split_boxes(int level, size_t bytes_per_box) {
  const size_t b = (size_t)m2l_split_most(level, bytes_per_box) << (3 * level);
  return b < 32768 ? b : 32768;
}

// The same for the run-time-order Helmholtz kernels.  M2L: one block runs on a
// CU at a time (its LDS), and the offsets of a chunk of 8 targets are split
// until there are about three rounds of blocks; the split depends on the
// chunk count only.
inline int wide_nsplit(unsigned nchunks) {
  const unsigned s = nchunks ? 768 / nchunks : 1;
  return s < 1 ? 1 : s > 27 ? 27 : (int)s;
}
inline size_t wide_split_boxes(int level) {
  const size_t b = (size_t)27 << (3 * level);
  return b < 768 * 8 ? b : 768 * 8;
}
// M2M: a block per child digit while there are few parents
inline int wide_m2m_nsplit(unsigned nchunks) { return nchunks < 128 ? 8 : 1; }
inline size_t wide_m2m_boxes(int level) {
  const size_t b = (size_t)8 << (3 * level);
  return b < 8 * 8 * 127 ? b : 8 * 8 * 127;
}

}  // namespace wbfmm
