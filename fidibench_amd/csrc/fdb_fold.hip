// fdb_fold.hip -- the reference's sequential left fold of a field
// (std::accumulate, pletzer/fidibench upwind/cxx/upwind.cxx:91-103;
// Filter::computeCheckSum, cxx/Filter.cpp:466-485), in parallel on the
// device and with the same bits.
//
// s <- RN(s + x) is not associative, but while s stays inside one binade,
// |s| in [2^e, 2^(e+1)), it is arithmetic on integers: with u = 2^(e-52),
// m = |s|/u and t = sign(s)*x/u,
//     m <- m + RN(t),   a tie of t going to the neighbour that makes the
//                       new m even,
// so the effect of a run of values on m is one integer per parity of the m
// it starts from, and runs compose (FoldMap).  Three launches: the sum of
// every chunk of values in any order; their prefix sums, which guess s --
// and so its sign and binade -- at each chunk's start; and each chunk's
// map in that binade, with bounds on the m it passes through.  The host
// then walks the chunks with the true s: a chunk whose guess holds and
// whose bounds keep m inside the binade costs one integer add; any other
// (where s changes binade, some log2 of them in a field of one sign; at
// s = 0; values that are not finite) is folded value by value as the
// reference does, from a copy the third launch made of it.
//
// Bound: two reads of the field (HBM) and some 50 us of launches, copies
// and the values folded on the host, against the copy of the whole field
// over PCIe and one dependent host addition per value.  FP64 checksum
// before / now: 128^3 5.9 ms / 66 us, 256^3 59 ms / 0.19 ms, 512^3 388 ms /
// 0.88 ms (two passes at 2.4 TB/s); std, two folds, twice that.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>
#include <cstring>

#include "../../include/fidibench_amd/fdb_upwind.h"
#include "fdb_fold_map.h"
#include "fdb_internal.h"

#pragma clang fp contract(off)

namespace fdb {
namespace {

constexpr int kFoldThreads = 256;
constexpr int kFoldPer = 8;                               // consecutive values per thread
constexpr int kFoldTile = kFoldThreads * kFoldPer;        // values staged in LDS at a time
constexpr uint64_t kFoldMaxChunks = 16384;
constexpr size_t kFoldGatherBytes = 16u << 20;            // chunks copied out, at most
constexpr double kTwo52 = 4503599627370496.0;

__device__ inline double fold_ld(const double* x, uint64_t i) { return x[i]; }
__device__ inline double fold_ld(const float* x, uint64_t i) { return (double)x[i]; }
__device__ inline double fold_ld(const uint16_t* x, uint64_t i) {
  return (double)__builtin_bit_cast(float, (uint32_t)x[i] << 16);
}

// The folded term of a field value: the value (checksum) or its squared
// distance from the mean (std).
struct FoldTerm {
  int squares;
  double mean;
  __device__ double operator()(double f) const {
    if (!squares) return f;
    const double d = f - mean;
    return d * d;
  }
};

template <typename TS>
__global__ __launch_bounds__(kFoldThreads) void fold_sum_kernel(const TS* __restrict__ x,
                                                                uint64_t n, uint64_t chunk,
                                                                FoldTerm term,
                                                                double* __restrict__ sums) {
  __shared__ double red[kFoldThreads / 64];
  const uint64_t b = (uint64_t)blockIdx.x * chunk;
  const uint64_t e = b + chunk < n ? b + chunk : n;
  double s = 0.0;
  uint64_t i = b + threadIdx.x;
  for (; i + (kFoldPer - 1) * kFoldThreads < e; i += kFoldTile) {
    double v[kFoldPer];
#pragma unroll
    for (int k = 0; k < kFoldPer; ++k) v[k] = term(fold_ld(x, i + (uint64_t)k * kFoldThreads));
#pragma unroll
    for (int k = 0; k < kFoldPer; ++k) s += v[k];
  }
  for (; i < e; i += kFoldThreads) s += term(fold_ld(x, i));
  for (int w = 32; w > 0; w >>= 1) s += __shfl_down(s, w);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) sums[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

// starts[c] = sums[0] + .. + sums[c-1], in place; one block.  Clears the
// count of copied chunks too.
__global__ __launch_bounds__(1024) void fold_scan_kernel(double* __restrict__ sums, int nchunks,
                                                         unsigned* __restrict__ copied) {
  __shared__ double part[1024];
  const int t = threadIdx.x;
  const int per = (nchunks + 1023) / 1024;
  const int b = t * per, e = b + per < nchunks ? b + per : nchunks;
  double s = 0.0;
  for (int i = b; i < e; ++i) s += sums[i];
  part[t] = s;
  __syncthreads();
  for (int w = 1; w < 1024; w <<= 1) {
    const double v = t >= w ? part[t - w] : 0.0;
    __syncthreads();
    part[t] += v;
    __syncthreads();
  }
  double run = t > 0 ? part[t - 1] : 0.0;
  for (int i = b; i < e; ++i) {
    const double v = sums[i];
    sums[i] = run;
    run += v;
  }
  if (t == 0) *copied = 0;
}

// One block per chunk: its FoldMap in the guessed binade, or a copy of its
// terms for the host where no single binade can hold (see FoldRec).
template <typename TS>
__global__ __launch_bounds__(kFoldThreads) void fold_map_kernel(
    const TS* __restrict__ x, uint64_t n, uint64_t chunk, FoldTerm term,
    const double* __restrict__ starts, FoldRec* __restrict__ recs, unsigned* __restrict__ copied,
    double* __restrict__ gather, unsigned slots) {
  // A thread's kFoldPer consecutive values are kFoldPer + 1 apart in LDS.
  __shared__ double vals[kFoldTile + kFoldThreads];
  __shared__ FoldMap wave_map[kFoldThreads / 64];
  __shared__ int any_bad, any_value;
  __shared__ unsigned slot;
  const int t = threadIdx.x;
  const uint64_t b = (uint64_t)blockIdx.x * chunk;
  const uint64_t e = b + chunk < n ? b + chunk : n;
  const double s0 = starts[blockIdx.x];
  const int neg = __builtin_signbit(s0) ? 1 : 0;
  // (ilogb of 0, Inf and NaN is out of the range tested.)
  const int ex = ilogb(s0);
  bool bad = !(ex >= -1021 && ex <= 1022);
  const int scale = bad ? 0 : 52 - ex;
  if (t == 0) {
    any_bad = 0;
    any_value = 0;
  }
  FoldMap run = fold_identity();  // of the chunk's tiles so far (thread 0)
  bool value = false;
  for (uint64_t tb = b; tb < e; tb += kFoldTile) {
#pragma unroll
    for (int k = 0; k < kFoldPer; ++k) {
      const int j = t + k * kFoldThreads;
      const uint64_t i = tb + (uint64_t)j;
      const double v = i < e ? term(fold_ld(x, i)) : 0.0;
      value |= v != 0.0;
      vals[j + j / kFoldPer] = neg ? -v : v;
    }
    __syncthreads();
    FoldMap m = fold_identity();
#pragma unroll
    for (int k = 0; k < kFoldPer; ++k) {
      const double v = ldexp(vals[t * (kFoldPer + 1) + k], scale);
      bad |= !(fabs(v) < kTwo52);
      fold_append(m, v);
    }
    // Ordered reduction over the wave, then over the waves.
    for (int w = 1; w < 64; w <<= 1) {
      const FoldMap o = {__shfl_down(m.d0, w), __shfl_down(m.d1, w), __shfl_down(m.lo, w),
                         __shfl_down(m.hi, w)};
      m = fold_then(m, o);  // (lanes that are no multiple of 2w hold leftovers)
    }
    if ((t & 63) == 0) wave_map[t >> 6] = m;
    __syncthreads();
    if (t == 0)
      for (int w = 0; w < kFoldThreads / 64; ++w) run = fold_then(run, wave_map[w]);
  }
  if (bad) any_bad = 1;
  if (value) any_value = 1;
  __syncthreads();
  if (t == 0) {
    FoldRec rec;
    rec.d0 = run.d0;
    rec.d1 = run.d1;
    rec.lo = run.lo;
    rec.hi = run.hi;
    rec.ex = ex;
    rec.neg = neg;
    rec.slot = -1;
    const double m0 = ldexp(fabs(s0), scale);
    const bool fits = !any_bad && fold_fits(m0, rec.lo, rec.hi, fold_slack(n));
    rec.kind = !any_value ? kFoldZero : (fits ? kFoldMapped : kFoldRaw);
    slot = slots;
    if (rec.kind == kFoldRaw) {
      slot = atomicAdd(copied, 1u);
      if (slot < slots) rec.slot = (int)slot;
    }
    recs[blockIdx.x] = rec;
  }
  __syncthreads();
  if (slot < slots) {
    double* g = gather + (uint64_t)slot * chunk;
    for (uint64_t i = b + t; i < e; i += kFoldThreads) g[i - b] = term(fold_ld(x, i));
  }
}

double fold_values(double s, const double* v, uint64_t n) {
  for (uint64_t i = 0; i < n; ++i) s = s + v[i];
  return s;
}

}  // namespace

FoldPlan fold_plan(uint64_t n) {
  FoldPlan p;
  p.n = n;
  const uint64_t per = (n + kFoldMaxChunks - 1) / kFoldMaxChunks;
  p.chunk = std::max<uint64_t>(1, (per + kFoldTile - 1) / kFoldTile) * kFoldTile;
  p.nchunks = (n + p.chunk - 1) / p.chunk;
  // Chunks that can be copied out: all of them up to kFoldGatherBytes (fields
  // whose sum keeps passing through zero have no others, and fold on the host
  // from the copies), else a quarter.
  const uint64_t most = kFoldGatherBytes / (p.chunk * sizeof(double));
  p.slots = p.nchunks <= most ? p.nchunks
                              : std::max<uint64_t>(8, std::min<uint64_t>(p.nchunks / 4 + 16, most));
  // [count | records | copied chunks | prefix sums]
  p.rec_off = 64;
  p.gather_off = (p.rec_off + p.nchunks * sizeof(FoldRec) + 63) / 64 * 64;
  p.host_bytes = p.gather_off + p.slots * p.chunk * sizeof(double);
  p.dev_bytes = p.host_bytes + p.nchunks * sizeof(double);
  return p;
}

hipError_t fold_exact(int dtype, const void* x, const FoldPlan& p, bool squares, double mean,
                      char* dev, char* host, hipStream_t s, double* out, bool* done) {
  *done = false;
  unsigned* copied = reinterpret_cast<unsigned*>(dev);
  FoldRec* recs = reinterpret_cast<FoldRec*>(dev + p.rec_off);
  double* gather = reinterpret_cast<double*>(dev + p.gather_off);
  double* sums = reinterpret_cast<double*>(dev + p.host_bytes);
  const FoldTerm term{squares ? 1 : 0, mean};
  const dim3 grid((unsigned)p.nchunks), block(kFoldThreads);
#define FDB_FOLD(TS)                                                                            \
  hipLaunchKernelGGL(fold_sum_kernel<TS>, grid, block, 0, s, (const TS*)x, p.n, p.chunk, term,  \
                     sums);                                                                     \
  hipLaunchKernelGGL(fold_scan_kernel, dim3(1), dim3(1024), 0, s, sums, (int)p.nchunks, copied); \
  hipLaunchKernelGGL(fold_map_kernel<TS>, grid, block, 0, s, (const TS*)x, p.n, p.chunk, term,  \
                     sums, recs, copied, gather, (unsigned)p.slots)
  switch (storage_dtype(dtype)) {
    case FDB_F64: FDB_FOLD(double); break;
    case FDB_F32: FDB_FOLD(float); break;
    case FDB_BF16: FDB_FOLD(uint16_t); break;
    default: return hipErrorInvalidValue;
  }
#undef FDB_FOLD
  if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
  // The records with the first copied chunks, in one transfer; the others
  // if there are any.
  const uint64_t slot_bytes = p.chunk * sizeof(double);
  const uint64_t first = std::min<uint64_t>(p.slots, std::max<uint64_t>(1, (512u << 10) / slot_bytes));
  if (hipError_t e = hipMemcpyAsync(host, dev, p.gather_off + first * slot_bytes,
                                    hipMemcpyDeviceToHost, s);
      e != hipSuccess)
    return e;
  if (hipError_t e = hipStreamSynchronize(s); e != hipSuccess) return e;
  unsigned count;
  std::memcpy(&count, host, sizeof(count));
  if (count > p.slots) return hipSuccess;  // too many: the caller folds the whole field
  if (count > first) {
    const uint64_t off = p.gather_off + first * slot_bytes;
    if (hipError_t e = hipMemcpyAsync(host + off, dev + off, (count - first) * slot_bytes,
                                      hipMemcpyDeviceToHost, s);
        e != hipSuccess)
      return e;
    if (hipError_t e = hipStreamSynchronize(s); e != hipSuccess) return e;
  }
  const FoldRec* rec = reinterpret_cast<const FoldRec*>(host + p.rec_off);
  const double* vals = reinterpret_cast<const double*>(host + p.gather_off);
  double acc = 0.0;
  for (uint64_t c = 0; c < p.nchunks; ++c) {
    if (!fold_step(rec[c], vals, p.chunk, std::min(p.chunk, p.n - c * p.chunk), &acc))
      return hipSuccess;  // a mapped chunk whose guess failed: the caller folds
  }
  *out = acc;
  *done = true;
  return hipSuccess;
}

bool fold_step(const FoldRec& r, const double* vals, uint64_t chunk, uint64_t cnt, double* s) {
  if (r.kind == kFoldZero) return true;  // s + (+-0) is s (s is never -0: it starts at +0)
  if (r.kind == kFoldRaw) {
    if (r.slot < 0) return false;
    *s = fold_values(*s, vals + (uint64_t)r.slot * chunk, cnt);
    return true;
  }
  uint64_t bits;
  std::memcpy(&bits, s, sizeof(bits));
  const int e = (int)((bits >> 52) & 0x7ff) - 1023;
  if (e != r.ex || (int)(bits >> 63) != r.neg) return false;
  const uint64_t low = (1ull << 52) - 1;
  const int64_t m = (int64_t)((bits & low) | (1ull << 52));
  // Strictly inside the binade after every value (lo and hi are exact
  // below 2^53; beyond that the comparison fails either way).
  if (!((double)m + r.lo >= kTwo52 + 2.0 && (double)m + r.hi <= 2.0 * kTwo52 - 2.0)) return false;
  const int64_t m1 = m + (int64_t)((m & 1) ? r.d1 : r.d0);
  bits = (bits & ~low) | ((uint64_t)m1 & low);
  std::memcpy(s, &bits, sizeof(bits));
  return true;
}

}  // namespace fdb
