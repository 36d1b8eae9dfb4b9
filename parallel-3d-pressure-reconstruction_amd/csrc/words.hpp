// Source iteration over merged words (words.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "kernels.hpp"

namespace omni3d {

// Rows (sources) in groups of consecutive rows, one workgroup of `chunks`
// wavefronts each; a group's entries sorted by source, one word per entry or
// per 1, 2 or 4 equal ones: row in group << word_row_shift(chunks) | source << 2
// | log2 of the multiplicity.  A wavefront takes blocks of 256 words, 4 per
// lane with one 16-byte load: word u of lane l is the block's entry 64 u + l,
// so that one gather serves 64 consecutive entries, a few 128-byte lines.  The
// last row number of a group is no row's: the words that fill up a group's
// last block point at it.
constexpr int word_rows(int chunks) { return 64 * chunks - 1; }
constexpr int word_row_shift(int chunks) { return chunks == 8 ? 23 : 24; }
constexpr int word_max_sources(int chunks) { return 1 << (word_row_shift(chunks) - 2); }
constexpr int kWordBlock = 256;

// Device pointers of the layout.
struct WordMat {
  int nS = 0;
  int G = 0;       // groups
  int chunks = 8;  // wavefronts per group, 4 or 8
  const int* grow = nullptr;            // [G + 1] first row of each group
  const unsigned int* bptr = nullptr;   // [G + 1] first block of each group
  const unsigned int* words = nullptr;  // [(bptr[G] + 1) * 256], the last of no row
  const uint4* dc = nullptr;            // [nS] (diagonal, visit count, entries, 0)
};

// One reconstruction's iteration: iteration k reads pb[(k - 1) & 1] and
// writes pb[k & 1].  With srow the increment form (FP32 ray sums): srow[nS]
// FP64 row sums kept across iterations, db the FP32 increments in turn.
struct WordIter {
  WordMat m;
  const int* slist = nullptr;
  const long long* bs = nullptr;
  const double* pinit = nullptr;
  int seed = 0;
  int first = 0;  // first workgroup of a multi-snapshot launch
  double* pb[2] = {nullptr, nullptr};
  double* srow = nullptr;
  float* db[2] = {nullptr, nullptr};
  DevScalars* sc = nullptr;
  double* part = nullptr;  // word_part_bytes(G): sums and max of two iterations
};
constexpr size_t word_part_bytes(int G) { return sizeof(double) * 6 * (size_t)(G > 0 ? G : 1); }

// iteration k (1 .. max_iter); launch_words_finish ends the loop
hipError_t launch_iterate_words(int k, const WordIter& it, double tol, hipStream_t st);
hipError_t launch_iterate_words_multi(int chunks, bool inc, int k, const WordIter* desc,
                                      const unsigned int* blk_snap, unsigned int nblocks,
                                      double tol, hipStream_t st);
hipError_t launch_words_finish(int k, const WordIter& it, int max_iter, double tol, hipStream_t st);

// Builder: from the sorted (group << 32 | source << rb | row) keys the merged
// words' flags, their exclusive sums per entry (by the caller), the groups'
// first words and block counts (nblk[G] = 0), and the words.
hipError_t launch_word_flags(int64_t n, const unsigned long long* keys, unsigned int* flag,
                             hipStream_t st);
hipError_t launch_word_blocks(int G, const int* grow, const unsigned long long* rowptr, int64_t n,
                              const unsigned int* excl, unsigned int nwords, unsigned int* wfirst,
                              unsigned int* nblk, hipStream_t st);
hipError_t launch_word_write(int64_t n, int chunks, const unsigned long long* keys,
                             const unsigned int* flag, const unsigned int* excl,
                             const unsigned int* wfirst, const unsigned int* bptr,
                             unsigned int nblocks, unsigned int* words, hipStream_t st);
hipError_t launch_word_rowdata(int nS, const unsigned long long* rowptr, const unsigned int* diag,
                               const unsigned int* cnt, const int* slist, uint4* dc,
                               hipStream_t st);

}  // namespace omni3d
