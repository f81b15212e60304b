// fdb_plane.hip -- one or several upwind steps of a 2-D field in one pass
// over memory (Upwind<2>, pletzer/fidibench upwind/cxx/upwind.cxx:64-84; the
// 3-D pass is tb_kernel in fdb_kernels.hip).
//
// A wave owns 64 lanes x 2 consecutive columns, H = K rounded up to even of
// them halo on the upwind side, and marches along axis 1 from upwind to
// downwind; at every row it computes levels 1..K in registers.  Level l of
// a row needs level l-1 of that row -- its own two columns and one of the
// neighbouring lane (a DPP move) -- and of the row before it (kept per level
// in prev).  It starts K rows before its chunk, so every level is valid
// when output begins.  With no second tile axis there is nothing to
// exchange between waves: no LDS and no barrier.  Each value is produced by
// the operations of K one-step launches on the same inputs, in their
// order, and rounded through the storage type, so the bits are the same.
//
// Bound: vector-ALU issue (6 operations and one 64-bit lane move per two
// cells and level) where the fields fit the Infinity Cache, HBM beyond it.
// 2000 x 3000 FP64: 8 steps 21.8 us, 2.7 us a step against 14.6 one step
// per launch; 8000 x 8000 FP64 (HBM) 25.4 us a step against 180.  Two
// columns per lane measured 21.8 us against 25.8 with one (more halo and
// lane moves) and 27.4 with four (fewer waves); a prefetch of two rows 21.8
// against 24.1 with four (the loop no longer fits well).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "../../include/fidibench_amd/fdb_upwind.h"
#include "fdb_internal.h"

#pragma clang fp contract(off)

namespace fdb {
namespace {

constexpr int kCols = 2;          // columns per lane
constexpr int kWidth = 64 * kCols;
constexpr int kWaves = 4;         // independent waves per block
// Rows loaded ahead.  One step: all rows of a chunk (kStepChunk and the
// one before it), so a wave has its whole work in flight at once.
constexpr int prefetch(int k) { return k == 1 ? 4 : 2; }
constexpr int kStepChunk = prefetch(1) - 1;

using u32x2 = uint32_t __attribute__((ext_vector_type(2)));
using u32x4 = uint32_t __attribute__((ext_vector_type(4)));

// Storage type: arithmetic type, and two adjacent values as one access.
template <typename TS> struct Cell;
template <> struct Cell<double> {
  using M = double;
  using Pair = u32x4;
  __device__ static M rnd(M x) { return x; }
  __device__ static void ld2(__amdgpu_buffer_rsrc_t rs, uint32_t o, M (&x)[2]) {
    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rs, o, 0, 0);
    x[0] = __builtin_bit_cast(double, u32x2{v.x, v.y});
    x[1] = __builtin_bit_cast(double, u32x2{v.z, v.w});
  }
  __device__ static M ld(__amdgpu_buffer_rsrc_t rs, uint32_t o) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rs, o, 0, 0));
  }
  template <int AUX>
  __device__ static void st2(const M (&x)[2], __amdgpu_buffer_rsrc_t rs, uint32_t o) {
    const u32x2 a = __builtin_bit_cast(u32x2, x[0]), b = __builtin_bit_cast(u32x2, x[1]);
    __builtin_amdgcn_raw_buffer_store_b128(u32x4{a.x, a.y, b.x, b.y}, rs, o, 0, AUX);
  }
  template <int AUX> __device__ static void st(M x, __amdgpu_buffer_rsrc_t rs, uint32_t o) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, x), rs, o, 0, AUX);
  }
};
template <> struct Cell<float> {
  using M = float;
  __device__ static M rnd(M x) { return x; }
  __device__ static void ld2(__amdgpu_buffer_rsrc_t rs, uint32_t o, M (&x)[2]) {
    const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(rs, o, 0, 0);
    x[0] = __builtin_bit_cast(float, (uint32_t)v.x);
    x[1] = __builtin_bit_cast(float, (uint32_t)v.y);
  }
  __device__ static M ld(__amdgpu_buffer_rsrc_t rs, uint32_t o) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, o, 0, 0));
  }
  template <int AUX>
  __device__ static void st2(const M (&x)[2], __amdgpu_buffer_rsrc_t rs, uint32_t o) {
    __builtin_amdgcn_raw_buffer_store_b64(
        u32x2{__builtin_bit_cast(uint32_t, x[0]), __builtin_bit_cast(uint32_t, x[1])}, rs, o, 0,
        AUX);
  }
  template <int AUX> __device__ static void st(M x, __amdgpu_buffer_rsrc_t rs, uint32_t o) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, x), rs, o, 0, AUX);
  }
};
template <> struct Cell<uint16_t> {  // bf16 storage, round to nearest even
  using M = float;
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  __device__ static M widen(uint32_t h) { return __builtin_bit_cast(float, h << 16); }
  // The pair (+0, x) to bf16: the binary32 value of bf16(x).
  __device__ static M rnd(M x) {
    return __builtin_bit_cast(float, __builtin_convertvector(f2{0.0f, x}, b2));
  }
  __device__ static void ld2(__amdgpu_buffer_rsrc_t rs, uint32_t o, M (&x)[2]) {
    const uint32_t v = __builtin_amdgcn_raw_buffer_load_b32(rs, o, 0, 0);
    x[0] = widen(v & 0xffffu);
    x[1] = widen(v >> 16);
  }
  __device__ static M ld(__amdgpu_buffer_rsrc_t rs, uint32_t o) {
    return widen((uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rs, o, 0, 0));
  }
  // (Stored values have been through rnd: the low halves are zero.)
  template <int AUX>
  __device__ static void st2(const M (&x)[2], __amdgpu_buffer_rsrc_t rs, uint32_t o) {
    __builtin_amdgcn_raw_buffer_store_b32(
        (__builtin_bit_cast(uint32_t, x[0]) >> 16) | __builtin_bit_cast(uint32_t, x[1]), rs, o, 0,
        AUX);
  }
  template <int AUX> __device__ static void st(M x, __amdgpu_buffer_rsrc_t rs, uint32_t o) {
    __builtin_amdgcn_raw_buffer_store_b16((uint16_t)(__builtin_bit_cast(uint32_t, x) >> 16), rs,
                                          o, 0, AUX);
  }
};

// The neighbouring lane's value (+-1 lane; the edge lane's is a halo
// column's, where any value is harmless).
template <int CTRL, typename T>
__device__ inline T lane_shift(T x) {
  constexpr int W = sizeof(T) / 4;
  struct Words { int w[W]; };
  Words a = __builtin_bit_cast(Words, x), r;
#pragma unroll
  for (int i = 0; i < W; ++i) r.w[i] = __builtin_amdgcn_mov_dpp(a.w[i], CTRL, 0xf, 0xf, true);
  return __builtin_bit_cast(T, r);
}

__device__ inline int64_t mod(int64_t x, int64_t n) {
  x %= n;
  return x < 0 ? x + n : x;
}

struct PlaneArgs {
  int64_t n1, n2;
  int u1;          // upwind side of the marched axis
  int64_t chunk, tiles2, ntiles;
};

template <typename TS>
__device__ inline __amdgpu_buffer_rsrc_t row_of(const TS* p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<TS*>(p), 0, bytes, 0x00020000);
}

// LO2: the axis-2 neighbour is column c-1.  PAIRS: an even n2 and aligned
// fields, so a lane's two columns are one access (the wrap never parts
// them).  NT: streaming stores.  Every memory access is unconditional --
// columns and rows that are not output are dropped by the store's range
// check -- so the compiler can count the outstanding ones and the loads
// stay two rows ahead.
template <typename TS, int K, bool LO2, bool PAIRS, bool NT>
__global__ __launch_bounds__(64 * kWaves) void plane_kernel(const TS* __restrict__ in,
                                                            TS* __restrict__ out, PlaneArgs a,
                                                            typename Cell<TS>::M c1,
                                                            typename Cell<TS>::M c2) {
  using C = Cell<TS>;
  using M = typename C::M;
  constexpr int H = K + (K & 1), AUX = NT ? 2 : 0, kPrefetch = prefetch(K);
  constexpr uint32_t kDropped = 0x7ffffff0u;  // past any row's end
  int64_t t = blockIdx.x;
  {  // blocks go to the 8 XCDs in turn: a contiguous range of tiles for each
    const int64_t x = t & 7, q = gridDim.x >> 3, r = gridDim.x & 7;
    t = x * q + (x < r ? x : r) + (t >> 3);
  }
  const int lane = threadIdx.x;
  const int64_t tile = t * kWaves + __builtin_amdgcn_readfirstlane(threadIdx.y);
  if (tile >= a.ntiles) return;  // whole wave
  const int64_t t2 = tile % a.tiles2, ch = tile / a.tiles2;

  const int64_t o2 = t2 * (kWidth - H);  // first output column
  const int rbytes = (int)(a.n2 * (int64_t)sizeof(TS));
  uint32_t lo[kCols], so[kCols];  // byte offsets in a row: loads, stores
#pragma unroll
  for (int v = 0; v < kCols; ++v) {
    const int i = lane * kCols + v;
    const int64_t c = (LO2 ? o2 - H : o2) + i;  // unwrapped column
    lo[v] = (uint32_t)mod(c, a.n2) * (uint32_t)sizeof(TS);
    so[v] = ((LO2 ? i >= H : i < kWidth - H) && c < a.n2) ? lo[v] : kDropped;
  }
  const int64_t p_lo = ch * a.chunk;
  const int64_t p_hi = p_lo + a.chunk < a.n1 ? p_lo + a.chunk : a.n1;
  const int64_t step = a.u1 < 0 ? 1 : -1;
  const int cnt = (int)(p_hi - p_lo) + K;
  int64_t pw = mod(a.u1 < 0 ? p_lo - K : p_hi - 1 + K, a.n1);  // row computed
  int64_t pl = pw;                                             // row loaded next
  auto next = [&](int64_t p) {
    p += step;
    return p < 0 ? a.n1 - 1 : (p == a.n1 ? 0 : p);
  };
  auto load = [&](M (&x)[kCols]) {
    const __amdgpu_buffer_rsrc_t rs = row_of(in + pl * a.n2, rbytes);
    if constexpr (PAIRS) {
      C::ld2(rs, lo[0], x);
    } else {
#pragma unroll
      for (int v = 0; v < kCols; ++v) x[v] = C::ld(rs, lo[v]);
    }
    pl = next(pl);
  };

  M prev[K][kCols], ahead[kPrefetch][kCols];
#pragma unroll
  for (int l = 0; l < K; ++l)
#pragma unroll
    for (int v = 0; v < kCols; ++v) prev[l][v] = M(0);
#pragma unroll
  for (int u = 0; u < kPrefetch; ++u) load(ahead[u]);
  // (The rows of a last, partial trip are computed and dropped.)
  for (int m = 0; m < cnt; m += kPrefetch) {
#pragma unroll
    for (int u = 0; u < kPrefetch; ++u) {
      M x[kCols];
#pragma unroll
      for (int v = 0; v < kCols; ++v) x[v] = ahead[u][v];
      load(ahead[u]);
#pragma unroll
      for (int l = 0; l < K; ++l) {
        const M e = LO2 ? lane_shift<0x138>(x[kCols - 1]) : lane_shift<0x130>(x[0]);
        M g[kCols];
#pragma unroll
        for (int v = 0; v < kCols; ++v) {
          const M n2 = LO2 ? (v > 0 ? x[0] : e) : (v + 1 < kCols ? x[kCols - 1] : e);
          const M q1 = c1 * (prev[l][v] - x[v]);
          const M q2 = c2 * (n2 - x[v]);
          g[v] = x[v] - q1;
          g[v] = g[v] - q2;
        }
#pragma unroll
        for (int v = 0; v < kCols; ++v) {
          prev[l][v] = x[v];
          x[v] = C::rnd(g[v]);
        }
      }
      const int row = m + u;
      const __amdgpu_buffer_rsrc_t rs =
          row_of(out + pw * a.n2, row >= K && row < cnt ? rbytes : 0);
      if constexpr (PAIRS) {
        C::template st2<AUX>(x, rs, so[0]);
      } else {
#pragma unroll
        for (int v = 0; v < kCols; ++v) C::template st<AUX>(x[v], rs, so[v]);
      }
      pw = next(pw);
    }
  }
}

constexpr int64_t kWaveSlots = 1024;  // one wave on each SIMD

// Rows per chunk.  A wave's time is its rows, K of them warm-up, times a
// row's: the latency of its K dependent levels (measured 1.3 times one
// wave's issue), or the issue of all the waves on its SIMD.  Fields with
// more than eight waves per SIMD at 20 rows are bound by HBM, where short
// chunks measured best (8000 x 8000: 203 us at 20 rows, 229 at 64).
int64_t plane_chunk(const Grid3& g, int k, int64_t tiles2) {
  const int64_t n1 = g.n[1];
  if (k == 1) return std::min<int64_t>(kStepChunk, n1);
  auto waves = [&](int64_t c) { return tiles2 * ((n1 + c - 1) / c); };
  if (waves(20) > 8 * kWaveSlots) return std::min<int64_t>(20, n1);
  int64_t best = n1;
  double least = -1.0;
  for (int64_t c = std::min<int64_t>(4, n1); c <= std::min<int64_t>(n1, 512); ++c) {
    const int64_t rows = (c + k + prefetch(k) - 1) / prefetch(k) * prefetch(k);
    const double per = std::max(1.3, (double)((waves(c) + kWaveSlots - 1) / kWaveSlots));
    if (least < 0.0 || (double)rows * per < least) {
      least = (double)rows * per;
      best = c;
    }
  }
  return best;
}

PlaneArgs plane_args(const Grid3& g, int k) {
  PlaneArgs a;
  a.n1 = g.n[1];
  a.n2 = g.n[2];
  a.u1 = g.up[1];
  const int out = kWidth - (k + (k & 1));
  a.tiles2 = (a.n2 + out - 1) / out;
  a.chunk = plane_chunk(g, k, a.tiles2);
  a.ntiles = a.tiles2 * ((a.n1 + a.chunk - 1) / a.chunk);
  return a;
}

template <typename TS, int K>
hipError_t launch_k(const Grid3& g, const TS* src, TS* dst, hipStream_t s) {
  using M = typename Cell<TS>::M;
  const PlaneArgs a = plane_args(g, K);
  const int64_t blocks = (a.ntiles + kWaves - 1) / kWaves;
  if (blocks > 0x7fffffffLL) return hipErrorInvalidConfiguration;
  const bool pairs = a.n2 % 2 == 0 && ((uintptr_t)src | (uintptr_t)dst) % (2 * sizeof(TS)) == 0;
  // Stores stream past the caches once the two fields outgrow the Infinity
  // Cache (2000 x 3000 FP64 24 cached, 29 us streaming; 8000 x 8000 226, 203).
  const bool nt = 2 * g.ntot * (int64_t)sizeof(TS) > (256ll << 20);
  const bool lo2 = g.up[2] < 0;
  const M c1 = (M)g.c[1], c2 = (M)g.c[2];
  const dim3 grid((unsigned)blocks), block(64, kWaves);
#define FDB_PLANE(L, P, N)                                                                  \
  if (lo2 == L && pairs == P && nt == N)                                                    \
  hipLaunchKernelGGL((plane_kernel<TS, K, L, P, N>), grid, block, 0, s, src, dst, a, c1, c2)
  FDB_PLANE(false, false, false);
  FDB_PLANE(false, false, true);
  FDB_PLANE(false, true, false);
  FDB_PLANE(false, true, true);
  FDB_PLANE(true, false, false);
  FDB_PLANE(true, false, true);
  FDB_PLANE(true, true, false);
  FDB_PLANE(true, true, true);
#undef FDB_PLANE
  return hipGetLastError();
}

template <typename TS>
hipError_t launch_typed(const Grid3& g, const void* src, void* dst, int k, hipStream_t s) {
  const TS* in = (const TS*)src;
  TS* out = (TS*)dst;
  switch (k) {
    case 1:
      if constexpr (sizeof(TS) > 2) return launch_k<TS, 1>(g, in, out, s);
      return hipErrorNotSupported;
    case 2: return launch_k<TS, 2>(g, in, out, s);
    case 3: return launch_k<TS, 3>(g, in, out, s);
    case 4: return launch_k<TS, 4>(g, in, out, s);
    case 5: return launch_k<TS, 5>(g, in, out, s);
    case 6: return launch_k<TS, 6>(g, in, out, s);
    case 7: return launch_k<TS, 7>(g, in, out, s);
    case 8: return launch_k<TS, 8>(g, in, out, s);
    default: return hipErrorNotSupported;
  }
}

}  // namespace

// One step too where it is the faster launch, us by rows_kernel / here:
// FP64 2000 x 3000 24.7 / 14.6, 703 x 1214 6.5 / 4.0, 8000 x 8000 277 /
// 180; FP32 10.2 / 9.4, 5.7 / 3.6, 157 / 90; not bf16 (8.4 / 8.9, 56 / 61),
// whose 16-byte lanes there hold eight cells.
bool plane_pass_supported(int dtype, const Grid3& g, int k) {
  if (k < 1 || k > kMaxTimeBlock || !is_plane(g)) return false;
  if (dtype != FDB_F64 && dtype != FDB_F32 && (dtype != FDB_BF16 || k == 1)) return false;
  // 32-bit row offsets, below the one that marks a dropped store.
  return g.n[2] * (int64_t)dtype_size(dtype) < 0x7fffff00LL;
}

hipError_t launch_plane_pass(int dtype, const Grid3& g, const void* src, void* dst, int k,
                             hipStream_t s) {
  if (!plane_pass_supported(dtype, g, k)) return hipErrorNotSupported;
  switch (dtype) {
    case FDB_F64: return launch_typed<double>(g, src, dst, k, s);
    case FDB_F32: return launch_typed<float>(g, src, dst, k, s);
    default: return launch_typed<uint16_t>(g, src, dst, k, s);
  }
}

// Measured on 2000 x 3000 (FP64 17.7, 20.1 and 21.8 us for 4, 6 and 8
// steps, 14.6 for one; FP32 17.8, bf16 21.2 us for 8), 703 x 1213, 200 x
// 150 and 8000 x 8000: a launch, then the larger of its memory traffic and
// its waves' time.
float plane_pass_us(int dtype, const Grid3& g, int k) {
  const double bytes = 2.0 * (double)g.ntot * (double)dtype_size(dtype);
  const bool resident = bytes <= (double)(256ll << 20);
  if (k == 1 && dtype != FDB_F64 && dtype != FDB_F32) return rows_step_us(dtype, g);
  const PlaneArgs a = plane_args(g, k);
  if (k == 1) {  // ns per wave: 2077634 x 3, 1219781 x 1, 199464 x 3 (297, 175, 33 us FP64)
    const double waves = 1e-3 * (double)a.ntiles * (dtype == FDB_F64 ? 0.43 : 0.35);
    return (float)(3.0 + std::max(waves, bytes / (resident ? 8.3e6 : 5.7e6)));
  }
  const double level = dtype == FDB_F64 ? 0.0285 : (dtype == FDB_F32 ? 0.021 : 0.026);
  const double waves = (double)a.ntiles / (double)kWaveSlots;
  // (More than four waves per SIMD hide each other's latency: FP32 8000 x
  // 8000 8 steps 113 us, where the times at two waves add up to 145.)
  const double per = waves > 4.0 ? 0.75 * waves : std::max(1.3, waves);
  const double issue = (double)(a.chunk + k) * per * (0.03 + level * k);
  return (float)(4.0 + std::max(issue, bytes / (resident ? 7.0e6 : 5.0e6)));
}

}  // namespace fdb
