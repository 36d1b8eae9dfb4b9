// Source iteration over merged words: one iteration on the sources S,
// p_new[r] = (bs[r] + diag[r] p[r] + sum over r's entries of p[src]) / C[r]
// (kernel.cu:8840-8861 restricted to the voxels the rays read), and the
// layout it reads (words.hpp).
#include <hip/hip_runtime.h>

#include <cfloat>

#include "launch.hpp"
#include "walk.hpp"
#include "words.hpp"

namespace omni3d {

namespace {

using Quad = unsigned int __attribute__((ext_vector_type(4)));  // a 16-byte piece

// A load through the scalar cache (p uniform across the wavefront, written
// before this launch): independent ones travel together.
template <typename T>
__device__ __forceinline__ T sload(const T* p) {
  return *(const __attribute__((address_space(4))) T*)(uintptr_t)p;
}

// Reductions over a wavefront by DPP (within rows of 16, then across them;
// lanes without a partner take 0), the result given to all lanes.
template <int kCtrl>
__device__ __forceinline__ unsigned long long dpp64(unsigned long long x) {
  const unsigned int lo = (unsigned int)__builtin_amdgcn_update_dpp(
      0, (int)(unsigned int)x, kCtrl, 0xf, 0xf, true);
  const unsigned int hi = (unsigned int)__builtin_amdgcn_update_dpp(
      0, (int)(unsigned int)(x >> 32), kCtrl, 0xf, 0xf, true);
  return ((unsigned long long)hi << 32) | lo;
}
__device__ __forceinline__ unsigned long long last_lane(unsigned long long x) {
  const unsigned int lo = (unsigned int)__builtin_amdgcn_readlane((int)(unsigned int)x, 63);
  const unsigned int hi = (unsigned int)__builtin_amdgcn_readlane((int)(unsigned int)(x >> 32), 63);
  return ((unsigned long long)hi << 32) | lo;
}
__device__ __forceinline__ unsigned long long max64(unsigned long long a, unsigned long long b) {
  return a > b ? a : b;
}
__device__ __forceinline__ unsigned long long wave_max(unsigned long long x) {
  x = max64(x, dpp64<0x111>(x));
  x = max64(x, dpp64<0x112>(x));
  x = max64(x, dpp64<0x114>(x));
  x = max64(x, dpp64<0x118>(x));
  x = max64(x, dpp64<0x142>(x));
  x = max64(x, dpp64<0x143>(x));
  return last_lane(x);
}
__device__ __forceinline__ unsigned long long bits64(double x) {
  return (unsigned long long)__double_as_longlong(x);
}
__device__ __forceinline__ double f64(unsigned long long x) {
  return __longlong_as_double((long long)x);
}
__device__ __forceinline__ double wave_sum(double v) {
  v += f64(dpp64<0x111>(bits64(v)));
  v += f64(dpp64<0x112>(bits64(v)));
  v += f64(dpp64<0x114>(bits64(v)));
  v += f64(dpp64<0x118>(bits64(v)));
  v += f64(dpp64<0x142>(bits64(v)));
  v += f64(dpp64<0x143>(bits64(v)));
  return f64(last_lane(bits64(v)));
}

__device__ __forceinline__ double relative_change(double d2, double n2, double* num, double* den) {
  *num = sqrt(d2);
  *den = sqrt(n2);
  return *den > 0.0 ? *num / *den : (*num > 0.0 ? INFINITY : 0.0);
}

constexpr double kRoundBias = 6755399441055744.0;  // 1.5 * 2^52, as in to_fixed

// Iteration k of group g.  kInc 0: FP64 values gathered; 1: the first
// iteration of the increment form (p gathered, the row sums stored); 2: the
// FP32 increments gathered, their sums added to the row sums.
//
// What bounds it: 4.7 us of launch, load chain and reductions (160x128x96, all
// words left out), then the vector memory unit: a gather of 64 takes its 16
// cycles however few lines it touches, as does a 16-byte load of 64 words per
// lane (256^3: the return path is busy 27 of 34 us, the LDS adds 14 us, HBM and
// the cache beyond L2 7 TB/s of words).  Words of 2 bytes with shared bases,
// 100 MB for 159, needed one load more per 256 words and took 44 us for 34.
// Against words staged through LDS with bounds on each, sums and stop rule by
// the first workgroup and atomics, us per iteration: 32^3 5.0 for 7.8,
// 160x128x96 13.5 for 16.2, 256^3 FP32 34.3 for 37.6, 128^3 masked 15.7 for 18.4.
//
// A short launch is a chain of dependent loads (about 0.7 us each), so
// everything whose address is known travels together: one scalar round trip
// (ranges, stop flag), one vector one (the words, the rows' own values, the
// previous iteration's partial sums), the gathers.  Every workgroup reduces
// the previous iteration's partial sums itself -- its max |x| is the scale's,
// its relative change the stop rule's -- so that no counter is shared and a
// stopped iteration is known before anything is written.
template <int kG, int kInc>
__device__ __forceinline__ void iterate_words_body(const unsigned int g, const WordIter& q, int k,
                                                   double tol) {
  constexpr int kThreads = 64 * kG;
  constexpr int kRowShift = word_row_shift(kG);
  constexpr unsigned int kSrcField = ((1u << kRowShift) - 1u) & ~3u;
  __shared__ unsigned long long s_acc[kThreads];
  __shared__ double s_red[kG][2];
  __shared__ unsigned long long s_max[kG];
  const WordMat& m = q.m;
  DevScalars* __restrict__ sc = q.sc;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r0 = sload(&m.grow[g]), nr = sload(&m.grow[g + 1]) - r0;
  const unsigned int b0 = sload(&m.bptr[g]), b1 = sload(&m.bptr[g + 1]), fill = sload(&m.bptr[m.G]);
  const int stopped = sload(&sc->converged);
  const double inv = sload(&sc->inv_scale);
  const unsigned long long mx0 = sload(&sc->itmax_bits[0]);
  const double* __restrict__ pp = q.part + (size_t)((k - 1) & 1) * 3 * m.G;
  const int i0 = tid < m.G ? tid : 0, i1 = tid + kThreads < m.G ? tid + kThreads : 0;
  unsigned long long mx = bits64(pp[2 * m.G + i0]), mx1 = bits64(pp[2 * m.G + i1]);
  double d2 = 0.0, n2 = 0.0, d21 = 0.0, n21 = 0.0;
  if (tol > 0.0) {
    d2 = pp[i0];
    n2 = pp[m.G + i0];
    d21 = pp[i1];
    n21 = pp[m.G + i1];
  }
  // (before the loads whose places come with the flag: a stopped iteration)
  if (stopped) return;
  const double* __restrict__ pold = q.pb[(k - 1) & 1];
  double* __restrict__ pnew = q.pb[k & 1];
  const float* __restrict__ din = kInc == 2 ? q.db[(k - 1) & 1] : nullptr;
  // (loads at clamped places instead of under branches: they travel together)
  const Quad* __restrict__ w4 = reinterpret_cast<const Quad*>(m.words) + lane;
  unsigned int b = b0 + (unsigned int)wave;
  // (past the group's blocks: the filling block)
  auto block = [&](unsigned int i) { return w4[(size_t)(i < b1 ? i : fill) * 64]; };
  Quad c = block(b), d = block(b + kG);
  const int own = r0 + (tid < nr ? tid : 0);
  const double po = pold[own];
  const long long bv = q.bs[own];
  const Quad dc = reinterpret_cast<const Quad*>(m.dc)[own];
  double sr = 0.0;
  if constexpr (kInc == 2) sr = q.srow[own];
  s_acc[tid] = 0ull;
  if (k > 1) {
    // (the clamped loads repeat group 0: harmless in a max, left out of sums)
    mx = max64(mx, mx1);
    d2 = tid < m.G ? d2 : 0.0;
    n2 = tid < m.G ? n2 : 0.0;
    if (tid + kThreads < m.G) {
      d2 += d21;
      n2 += n21;
    }
    for (int i = tid + 2 * kThreads; i < m.G; i += kThreads) {
      mx = max64(mx, bits64(pp[2 * m.G + i]));
      if (tol > 0.0) {
        d2 += pp[i];
        n2 += pp[m.G + i];
      }
    }
    mx = wave_max(mx);
    if (tol > 0.0) {
      d2 = wave_sum(d2);
      n2 = wave_sum(n2);
    }
    if (lane == 0) {
      s_red[wave][0] = d2;
      s_red[wave][1] = n2;
      s_max[wave] = mx;
    }
  }
  __syncthreads();
  if (k > 1) {
    d2 = n2 = 0.0;
    mx = 0ull;
#pragma unroll
    for (int w = 0; w < kG; w++) {
      mx = max64(mx, s_max[w]);
      d2 += s_red[w][0];
      n2 += s_red[w][1];
    }
    if (tol > 0.0) {
      double num, den;
      const double rel = relative_change(d2, n2, &num, &den);
      if (rel < tol) {
        if (g == 0 && tid == 0) {
          sc->rel = rel;
          sc->dnum = num;
          sc->dden = den;
          sc->iter_done = k - 1;
          sc->converged = 1;
          sc->kstar = k - 1;
        }
        return;
      }
    }
  } else {
    mx = mx0;
  }
  const double B = f64(mx);
  const bool finite = B <= DBL_MAX;
  int ex = 0;
  (void)frexp(finite ? B : 1.0, &ex);
  ex = ex < -960 ? -960 : ex;  // (a tiny bound: keep the scale finite)
  const double scale = ldexp(1.0, 51 - ex), iscale = ldexp(1.0, ex - 51);
  for (; b < b1; b += 2 * kG) {
    const unsigned int w[8] = {c.x, c.y, c.z, c.w, d.x, d.y, d.z, d.w};
    double x[8];
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const unsigned int off = w[u] & kSrcField;
      if constexpr (kInc == 2)
        x[u] = (double)*reinterpret_cast<const float*>(reinterpret_cast<const char*>(din) + off);
      else
        x[u] = *reinterpret_cast<const double*>(reinterpret_cast<const char*>(pold) + 2u * off);
    }
    c = block(b + 2 * kG);
    d = block(b + 3 * kG);
    // every term rounded to the scale's unit (to_fixed; the product is exact,
    // the scale a power of two), times its multiplicity, an exact integer
    // sum: the same in any order and for any grouping.  The rounding bias
    // stays in, once per entry: the row's end takes it out.
#pragma unroll
    for (int u = 0; u < 8; u++)
      atomicAdd(&s_acc[w[u] >> kRowShift],
                bits64(__builtin_fma(x[u], scale, kRoundBias)) << (w[u] & 3u));
  }
  __syncthreads();
  d2 = n2 = 0.0;
  mx = 0ull;
  if (tid < nr) {
    double acc = (double)(long long)(s_acc[tid] - dc.z * bits64(kRoundBias)) * iscale;
    if (!finite) acc = B - B;
    if constexpr (kInc == 2) acc += sr;
    if constexpr (kInc != 0) q.srow[r0 + tid] = acc;
    double tot = (double)bv * inv + (double)dc.x * po + acc;
    if (k == 1 && q.seed && q.pinit) tot += q.pinit[q.slist[r0 + tid]];
    const double pn = dc.y > 0 ? tot / (double)dc.y : po;
    pnew[r0 + tid] = pn;
    const double df = pn - po;
    d2 = df * df;
    n2 = pn * pn;
    double mv = pn;
    if constexpr (kInc != 0) {
      const float dq = (float)df;
      q.db[k & 1][r0 + tid] = dq;
      mv = (double)dq;
    }
    mx = bits64(fabs(mv));
  }
  const int rw = (nr + 63) / 64;  // wavefronts with rows
  if (wave < rw) {
    d2 = wave_sum(d2);
    n2 = wave_sum(n2);
    mx = wave_max(mx);
    if (lane == 0) {
      s_red[wave][0] = d2;
      s_red[wave][1] = n2;
      s_max[wave] = mx;
    }
  }
  __syncthreads();
  if (tid == 0) {
    d2 = n2 = 0.0;
    mx = 0ull;
    for (int w = 0; w < rw; w++) {
      d2 += s_red[w][0];
      n2 += s_red[w][1];
      mx = max64(mx, s_max[w]);
    }
    double* __restrict__ pc = q.part + (size_t)(k & 1) * 3 * m.G;
    pc[g] = d2;
    pc[m.G + g] = n2;
    pc[2 * m.G + g] = f64(mx);
  }
}

template <int kG, int kInc>
__global__ void __launch_bounds__(64 * kG)
k_iterate_words(WordIter q, int k, double tol) {
  iterate_words_body<kG, kInc>(blockIdx.x, q, k, tol);
}

// Iteration k of many snapshots in one launch: workgroup b works for
// snapshot blk_snap[b] as its group b - first.
template <int kG, int kInc>
__global__ void __launch_bounds__(64 * kG)
k_iterate_words_multi(const WordIter* __restrict__ desc, const unsigned int* __restrict__ blk_snap,
                      int k, double tol) {
  const WordIter& q = desc[sload(&blk_snap[blockIdx.x])];
  iterate_words_body<kG, kInc>(blockIdx.x - (unsigned int)q.first, q, k, tol);
}

// Relative change of the last iteration k and the stop rule.
__global__ void __launch_bounds__(256)
k_words_finish(WordIter q, int k, int max_iter, double tol) {
  DevScalars* __restrict__ sc = q.sc;
  if (sc->converged) return;
  __shared__ double s[4][2];
  const int G = q.m.G, tid = threadIdx.x;
  const double* __restrict__ pp = q.part + (size_t)(k & 1) * 3 * G;
  double d2 = 0.0, n2 = 0.0;
  for (int i = tid; i < G; i += 256) {
    d2 += pp[i];
    n2 += pp[G + i];
  }
  d2 = wave_sum(d2);
  n2 = wave_sum(n2);
  if ((tid & 63) == 0) {
    s[tid >> 6][0] = d2;
    s[tid >> 6][1] = n2;
  }
  __syncthreads();
  if (tid == 0) {
    double num, den;
    const double rel = relative_change(((s[0][0] + s[1][0]) + s[2][0]) + s[3][0],
                                       ((s[0][1] + s[1][1]) + s[2][1]) + s[3][1], &num, &den);
    sc->rel = rel;
    sc->dnum = num;
    sc->dden = den;
    sc->iter_done = k;
    if ((tol > 0.0 && rel < tol) || k >= max_iter) {
      sc->converged = 1;
      sc->kstar = k;
    }
  }
}

// ---------------------------------------------------------------------------
// The layout.  A run of equal keys becomes words of multiplicity 4 as long as
// they fit, then 2, then 1.

__global__ void __launch_bounds__(256)
k_word_flags(int64_t n, const unsigned long long* __restrict__ k, unsigned int* __restrict__ flag) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int64_t c = 0;
  while (i - c - 1 >= 0 && k[i - c - 1] == k[i]) c++;
  // the third of a last three stands alone
  const bool third = (c & 3) == 2 && !(i + 1 < n && k[i + 1] == k[i]);
  flag[i] = (c & 3) == 0 || third ? 1u : 0u;
}

__global__ void __launch_bounds__(256)
k_word_blocks(int G, const int* __restrict__ grow, const unsigned long long* __restrict__ rowptr,
              int64_t n, const unsigned int* __restrict__ excl, unsigned int nwords,
              unsigned int* __restrict__ wfirst, unsigned int* __restrict__ nblk) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g > G) return;
  if (g == G) {
    nblk[g] = 0u;
    return;
  }
  auto first = [&](int h) {
    const unsigned long long pos = rowptr[grow[h]];
    return pos < (unsigned long long)n ? excl[pos] : nwords;
  };
  const unsigned int a = first(g), b = first(g + 1);
  wfirst[g] = a;
  nblk[g] = (b - a + kWordBlock - 1) / kWordBlock;
}

template <int kG>
__global__ void __launch_bounds__(256)
k_word_write(int64_t n, const unsigned long long* __restrict__ k,
             const unsigned int* __restrict__ flag, const unsigned int* __restrict__ excl,
             const unsigned int* __restrict__ wfirst, const unsigned int* __restrict__ bptr,
             unsigned int* __restrict__ words) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || !flag[i]) return;
  constexpr int rb = 32 - word_row_shift(kG);
  const unsigned long long key = k[i];
  unsigned int run = 1;  // equal keys from here on, up to 4 and up to the next word
  while (run < 4 && i + run < n && k[i + run] == key && !flag[i + run]) run++;
  const unsigned int g = (unsigned int)(key >> 32);
  const unsigned int row = (unsigned int)(key & ((1ull << rb) - 1ull));
  const unsigned int src = (unsigned int)(key >> rb) & ((1u << (32 - rb)) - 1u);
  const unsigned int at = excl[i] - wfirst[g], in = at % kWordBlock;
  const unsigned int slot = ((in & 63u) << 2) | (in >> 6);
  words[(size_t)bptr[g] * kWordBlock + (at - in) + slot] =
      (row << word_row_shift(kG)) | (src << 2) | (run == 4 ? 2u : run - 1u);
}

__global__ void __launch_bounds__(256)
k_word_rowdata(int nS, const unsigned long long* __restrict__ rowptr,
               const unsigned int* __restrict__ diag, const unsigned int* __restrict__ cnt,
               const int* __restrict__ slist, uint4* __restrict__ dc) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r < nS)
    dc[r] = uint4{diag ? diag[r] : 0u, cnt[slist[r]], (unsigned int)(rowptr[r + 1] - rowptr[r]), 0u};
}

unsigned int grid1(int64_t n) { return (unsigned int)((n + 255) / 256); }

}  // namespace

hipError_t launch_iterate_words(int k, const WordIter& it, double tol, hipStream_t st) {
  if (it.m.G < 1) return hipErrorInvalidValue;
#define OMNI_WORDS(C, I)                                                                       \
  hipLaunchKernelGGL((k_iterate_words<C, I>), dim3(it.m.G), dim3(64 * C), 0, st, it, k, tol)
  const int inc = it.srow ? (k == 1 ? 1 : 2) : 0;
  if (it.m.chunks == 8) {
    if (inc == 1) OMNI_WORDS(8, 1);
    else if (inc == 2) OMNI_WORDS(8, 2);
    else OMNI_WORDS(8, 0);
  } else {
    if (inc == 1) OMNI_WORDS(4, 1);
    else if (inc == 2) OMNI_WORDS(4, 2);
    else OMNI_WORDS(4, 0);
  }
#undef OMNI_WORDS
  return hipGetLastError();
}

hipError_t launch_iterate_words_multi(int chunks, bool incr, int k, const WordIter* desc,
                                      const unsigned int* blk_snap, unsigned int nblocks,
                                      double tol, hipStream_t st) {
#define OMNI_WORDS(C, I)                                                                     \
  hipLaunchKernelGGL((k_iterate_words_multi<C, I>), dim3(nblocks), dim3(64 * C), 0, st, desc,  \
                     blk_snap, k, tol)
  const int inc = incr ? (k == 1 ? 1 : 2) : 0;
  if (chunks == 8) {
    if (inc == 1) OMNI_WORDS(8, 1);
    else if (inc == 2) OMNI_WORDS(8, 2);
    else OMNI_WORDS(8, 0);
  } else {
    if (inc == 1) OMNI_WORDS(4, 1);
    else if (inc == 2) OMNI_WORDS(4, 2);
    else OMNI_WORDS(4, 0);
  }
#undef OMNI_WORDS
  return hipGetLastError();
}

hipError_t launch_words_finish(int k, const WordIter& it, int max_iter, double tol,
                               hipStream_t st) {
  hipLaunchKernelGGL(k_words_finish, dim3(1), dim3(256), 0, st, it, k, max_iter, tol);
  return hipGetLastError();
}

hipError_t launch_word_flags(int64_t n, const unsigned long long* keys, unsigned int* flag,
                             hipStream_t st) {
  hipLaunchKernelGGL(k_word_flags, dim3(grid1(n)), dim3(256), 0, st, n, keys, flag);
  return hipGetLastError();
}

hipError_t launch_word_blocks(int G, const int* grow, const unsigned long long* rowptr, int64_t n,
                              const unsigned int* excl, unsigned int nwords, unsigned int* wfirst,
                              unsigned int* nblk, hipStream_t st) {
  hipLaunchKernelGGL(k_word_blocks, dim3(grid1((int64_t)G + 1)), dim3(256), 0, st, G, grow, rowptr, n, excl,
                     nwords, wfirst, nblk);
  return hipGetLastError();
}

hipError_t launch_word_write(int64_t n, int chunks, const unsigned long long* keys,
                             const unsigned int* flag, const unsigned int* excl,
                             const unsigned int* wfirst, const unsigned int* bptr,
                             unsigned int nblocks, unsigned int* words, hipStream_t st) {
  const unsigned int fill = (unsigned int)(64 * chunks - 1) << word_row_shift(chunks);
  hipError_t e = launch_fill_u32(words, ((int64_t)nblocks + 1) * kWordBlock, fill, st);
  if (e != hipSuccess) return e;
  if (chunks == 8)
    hipLaunchKernelGGL(k_word_write<8>, dim3(grid1(n)), dim3(256), 0, st, n, keys, flag, excl,
                       wfirst, bptr, words);
  else
    hipLaunchKernelGGL(k_word_write<4>, dim3(grid1(n)), dim3(256), 0, st, n, keys, flag, excl,
                       wfirst, bptr, words);
  return hipGetLastError();
}

hipError_t launch_word_rowdata(int nS, const unsigned long long* rowptr, const unsigned int* diag,
                               const unsigned int* cnt, const int* slist, uint4* dc,
                               hipStream_t st) {
  hipLaunchKernelGGL(k_word_rowdata, dim3(grid1(nS)), dim3(256), 0, st, nS, rowptr, diag, cnt,
                     slist, dc);
  return hipGetLastError();
}

}  // namespace omni3d
