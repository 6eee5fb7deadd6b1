// Linear layers and row gathers around the attention path: the candle ops
// that surround Attention::attend in the reference's forward passes.
//   cev_linear      x . w^T (+ scale): Linear::forward of the q/k/v/o
//                   projections and the MLP (crates/cev-model/src/qwen3.rs:175-178,
//                   :229-233), the code head (crates/cev-model/src/engine.rs:463)
//                   and the d3 readout `answers.matmul(weight.t()) / temperature`
//                   (crates/cev-model/src/hybrid.rs:657).
//   cev_gather_rows table rows by index with a dtype conversion: Embedding
//                   rows (qwen3.rs:288-293), the gather of the answer rows
//                   (qwen3.rs:399, hybrid.rs:634), `to_dtype(F32)`
//                   (qwen3.rs:400) and the code head's rows of the tied
//                   embedding (engine.rs:155).
//
// Row counts of up to kRowsSmall (decode-like readouts, the code head of a
// few questions) run on this file's own kernel, which streams every weight
// row once, and f32 products that fill the chip on its split kernel (bf16
// matrix cores); all others are plain library GEMMs (hipBLASLt).  f32
// accumulation, the result rounded once to the output dtype as candle's
// matmul does.
#include <hipblaslt/hipblaslt-ext.hpp>
#include <hipblaslt/hipblaslt.h>

#include <cmath>
#include <map>
#include <mutex>
#include <string>
#include <tuple>
#include <type_traits>
#include <vector>

#include "cev_device.h"
#include "cev_internal.h"

namespace {

constexpr int kRowsSmall = 8;
constexpr int kLinWaves = 4;  // output columns per workgroup of the small-row kernel

template <typename T>
__device__ __forceinline__ float to_f32(T x);
template <>
__device__ __forceinline__ float to_f32<float>(float x) {
  return x;
}
template <>
__device__ __forceinline__ float to_f32<uint16_t>(uint16_t x) {
  return bf16_from_bits(x);
}

template <typename T>
__device__ __forceinline__ T from_f32(float x);
template <>
__device__ __forceinline__ float from_f32<float>(float x) {
  return x;
}
template <>
__device__ __forceinline__ uint16_t from_f32<uint16_t>(float x) {
  return bf16_bits(x);
}

struct LinArgs {
  const void* x;
  const void* w;
  void* y;
  int64_t m, n, k, ldx, ldw, ldy;
  float alpha;
};

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// One wave per output column j: the lanes stream w's row j in 16-byte
// chunks (read once), multiply it with each of the m <= MR input rows (hot
// in L2) and reduce across the wave.  f32 accumulation; k a multiple of the
// 16-byte chunk (checked by the launcher).  A lane's chunks are loaded NB at
// a time with clamped indices (rows past m read row m - 1, chunks past k the
// last chunk), so every load of a batch is unconditional and in flight
// together; only the accumulation skips them.  Each lane still adds its
// chunks in order.
template <typename T, typename TO, int MR, int NB>
__global__ __launch_bounds__(kLinWaves * 64) void linear_rows_kernel(LinArgs a) {
  constexpr int VEC = 16 / (int)sizeof(T);
  const int lane = threadIdx.x & 63;
  const int64_t j = (int64_t)blockIdx.x * kLinWaves + (threadIdx.x >> 6);
  if (j >= a.n) return;
  const T* wr = (const T*)a.w + j * a.ldw;
  float acc[MR];
#pragma unroll
  for (int r = 0; r < MR; ++r) acc[r] = 0.0f;
  for (int64_t e0 = (int64_t)lane * VEC; e0 < a.k; e0 += (int64_t)NB * 64 * VEC) {
    uint4 wv[NB], xv[MR][NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int64_t ec = min(e0 + (int64_t)b * 64 * VEC, a.k - VEC);
      wv[b] = *(const uint4*)(wr + ec);
#pragma unroll
      for (int r = 0; r < MR; ++r) xv[r][b] = *(const uint4*)((const T*)a.x + (int64_t)min(r, (int)a.m - 1) * a.ldx + ec);
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      if (e0 + (int64_t)b * 64 * VEC < a.k) {
        const T* w8 = (const T*)&wv[b];
#pragma unroll
        for (int r = 0; r < MR; ++r) {
          const T* x8 = (const T*)&xv[r][b];
#pragma unroll
          for (int i = 0; i < VEC; ++i) acc[r] = __builtin_fmaf(to_f32<T>(x8[i]), to_f32<T>(w8[i]), acc[r]);
        }
      }
    }
  }
#pragma unroll
  for (int r = 0; r < MR; ++r) {
    const float s = wave_sum(acc[r]);
    if (r < a.m && lane == 0) ((TO*)a.y)[r * a.ldy + j] = from_f32<TO>(s * a.alpha);
  }
}

// ---------------------------------------------------------------------------
// f32 products of more than kRowsSmall rows on the bf16 matrix cores.
// Every f32 value is split into three bf16 parts (round to nearest each; the
// parts' sum is the value, the second at most 2^-8 and the third 2^-17 of it)
// and six of the nine part products are summed in f32.  Of the three dropped
// ones the two larger are at most 2^-25 of the product each, all three 2^-24.
// Six bf16 products cost 6/16 of the f32 unit's time.  The products of the
// first parts have an accumulator of their own, rounded once per 16 products
// (the f32 unit's once per 2), and the five small ones, whose roundings weigh
// 2^-8 as much, another; they meet at the end.
//
// A workgroup of eight waves computes a 128 x 128 tile of y, each wave 64 x 32
// of it on 32x32x16 MFMAs.  A 32-deep slice of x and w goes through registers
// two slices ahead, is split there once for the whole workgroup while the
// slice before it is multiplied, and lies in LDS (two buffers of 48 KB) as
// three planes of 64-byte rows, 16-byte piece c of row r at c ^ (r / 4 % 4) so
// that a fragment read touches every bank.
// What bounds it: a slice takes 3000 clocks a CU where its MFMAs need 1536 and
// its LDS traffic (195 KB) 1500; 195-202 TFLOP/s of f32 products at 2048 rows
// (library 146-151).  Tried: one buffer and one slice ahead 134 us at
// 200 x 4096 x 2048 (72 now); four waves a tile 89; 64-wide tiles 113 against
// 95 at 912 x 4096 x 2048; 256 x 128 tiles 4-6 % faster at 2048 rows and half
// a round short at 912.
// Error against f64, N(0,1) x 0.02 N(0,1): 2.7e-7 at k = 2048 (library
// 8.1e-7), 4.9e-7 at 6144 (1.40e-6); with one accumulator for all six 7.0e-7
// and 1.24e-6 at the same times.
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

constexpr int kSliceK = 32;

constexpr int kSplitTile = 128, kSplitWaves = 8;

__global__ __launch_bounds__(kSplitWaves * 64) __attribute__((amdgpu_waves_per_eu(2))) void linear_split_kernel(LinArgs a, int parts) {
  constexpr int BM = kSplitTile, BN = kSplitTile, RP = kSplitWaves * 8;  // RP: rows per pass of the workgroup's loads
  constexpr int WM = BM / 2, WN = BN / (kSplitWaves / 2), TM = WM / 32, TN = WN / 32;
  constexpr int NX = BM / RP, NW = BN / RP;         // 16-byte loads per thread and slice
  constexpr int kPlane = (BM + BN) * kSliceK;       // one part of both operands, in bf16 values
  constexpr int kBuf = 3 * kPlane;                  // one slice
  __shared__ __align__(16) __bf16 lds[2 * kBuf];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n32 = lane & 31, u = lane >> 5, wm = wave & 1, wn = wave >> 1;
  // tiles of one XCD (workgroups go round-robin over the 8) are neighbours, m
  // fastest: they share w's rows
  const int total = gridDim.x, q8 = total / 8, r8 = total % 8, xcd = blockIdx.x % 8;
  const int mt = (int)((a.m + BM - 1) / BM), tiles = total / parts;
  int id = xcd * q8 + min(xcd, r8) + blockIdx.x / 8;
  const int part = id / tiles;
  id -= part * tiles;
  const int m0 = (id % mt) * BM, n0 = (id / mt) * BN;

  // this thread's rows (clamped) and column of a slice
  const int row = tid >> 3, c4 = (tid & 7) * 4;
  const float* xp[NX];
  const float* wp[NW];
#pragma unroll
  for (int i = 0; i < NX; ++i) xp[i] = (const float*)a.x + (int64_t)min(m0 + row + RP * i, (int)a.m - 1) * a.ldx;
#pragma unroll
  for (int i = 0; i < NW; ++i) wp[i] = (const float*)a.w + (int64_t)min(n0 + row + RP * i, (int)a.n - 1) * a.ldw;
  f32x4 xr[2][NX], wr[2][NW];  // two slices on their way
  auto load = [&](int k0, f32x4* xr, f32x4* wr) {
    // columns past k read the row's last four and count as zero
    const int k = k0 + c4, kc = min(k, (int)a.k - 4);
    const bool ok = k < (int)a.k;
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const f32x4 v = *(const f32x4*)(xp[i] + kc);
      xr[i] = ok ? v : f32x4{0, 0, 0, 0};
    }
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      const f32x4 v = *(const f32x4*)(wp[i] + kc);
      wr[i] = ok ? v : f32x4{0, 0, 0, 0};
    }
  };
  // row r of a plane (x's rows, then w's), 4 values at column c4
  auto put = [&](int buf, int r, const f32x4& v) {
    const int at = buf * kBuf + r * kSliceK + ((((c4 >> 3) ^ (r >> 2)) & 3) << 3) + (c4 & 4);
    f32x2 lo = {v[0], v[1]}, hi = {v[2], v[3]};
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const bf16x2 a2 = __builtin_convertvector(lo, bf16x2), b2 = __builtin_convertvector(hi, bf16x2);
      *(bf16x4*)(lds + i * kPlane + at) = bf16x4{a2[0], a2[1], b2[0], b2[1]};
      lo -= __builtin_convertvector(a2, f32x2);
      hi -= __builtin_convertvector(b2, f32x2);
    }
  };
  auto frag = [&](int buf, int plane, int r, int ks) {
    return *(const bf16x8*)(lds + buf * kBuf + plane * kPlane + r * kSliceK + ((((2 * ks + u) ^ (r >> 2)) & 3) << 3));
  };

  f32x16 acc[TM][TN], low[TM][TN];  // products of the first parts, and of the others
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = low[i][j] = f32x16{};
  // this part's slices of k
  const int all = (int)((a.k + kSliceK - 1) / kSliceK);
  const int s0 = (int)((int64_t)part * all / parts), s1 = (int)((int64_t)(part + 1) * all / parts);
  auto put_x = [&](int buf, const f32x4* v) {
#pragma unroll
    for (int i = 0; i < NX; ++i) put(buf, row + RP * i, v[i]);
  };
  auto put_w = [&](int buf, const f32x4* v) {
#pragma unroll
    for (int i = 0; i < NW; ++i) put(buf, BM + row + RP * i, v[i]);
  };
  auto multiply = [&](int buf, int ks) {
    bf16x8 fx[TM][3], fw[TN][3];
#pragma unroll
    for (int p = 0; p < 3; ++p) {
#pragma unroll
      for (int i = 0; i < TM; ++i) fx[i][p] = frag(buf, p, wm * WM + 32 * i + n32, ks);
#pragma unroll
      for (int j = 0; j < TN; ++j) fw[j][p] = frag(buf, p, BM + wn * WN + 32 * j + n32, ks);
    }
    // The first parts' product amid the others, whose accumulators then wait
    // less for each other (912 x 12288 x 2048 over changing weights: 268 us;
    // at the end 277, at the start 285, one accumulator for all 272).
#pragma unroll
    for (int q = 0; q < 6; ++q) {
      constexpr int kX[6] = {0, 1, 0, 2, 0, 1}, kW[6] = {2, 1, 0, 0, 1, 0};
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          f32x16& sum = kX[q] + kW[q] > 0 ? low[i][j] : acc[i][j];
          sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fx[i][kX[q]], fw[j][kW[q]], sum, 0, 0, 0);
        }
    }
  };
  // Slice sl is multiplied while slice sl + 1 is split into the other buffer
  // (past the end: a repeat of the last columns, counted as zero) and slices
  // sl + 2 and sl + 3 load.
  auto step = [&](int sl, auto buf_c) {
    constexpr int B = decltype(buf_c)::value, N = B ^ 1;
    multiply(B, 0);
    put_x(N, xr[N]);
    multiply(B, 1);
    put_w(N, wr[N]);
    load((sl + 3) * kSliceK, xr[N], wr[N]);
    __syncthreads();
  };
  load(s0 * kSliceK, xr[0], wr[0]);
  load((s0 + 1) * kSliceK, xr[1], wr[1]);
  put_x(0, xr[0]);
  put_w(0, wr[0]);
  load((s0 + 2) * kSliceK, xr[0], wr[0]);
  __syncthreads();
  for (int sl = s0; sl < s1; sl += 2) {
    step(sl, std::integral_constant<int, 0>{});
    if (sl + 1 < s1) step(sl + 1, std::integral_constant<int, 1>{});
  }

#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] += low[i][j];

  // An infinite value (or one above bf16's range) has no parts: x - bf16(x) is
  // not a number.  A wave whose quarter came out non-finite anywhere computes
  // it again in f32, one product after the other.
  float worst = 0.0f;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) worst += acc[i][j][e] * 0.0f;
  float* y = (float*)a.y + (int64_t)part * a.m * a.ldy;  // parts lie behind one another
  const int k0 = s0 * kSliceK, k1 = min(s1 * kSliceK, (int)a.k);
  if (__builtin_expect(__any(worst != 0.0f || worst != worst) != 0, 0)) {
#pragma unroll 1
    for (int e = lane; e < WM * WN; e += 64) {
      const int m = m0 + wm * WM + e / WN, n = n0 + wn * WN + e % WN;
      if (m >= a.m || n >= a.n) continue;
      const float* xq = (const float*)a.x + (int64_t)m * a.ldx;
      const float* wq = (const float*)a.w + (int64_t)n * a.ldw;
      float s = 0.0f;
#pragma unroll 1
      for (int k = k0; k < k1; ++k) s = __builtin_fmaf(xq[k], wq[k], s);
      y[(int64_t)m * a.ldy + n] = s * a.alpha;
    }
    return;
  }
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int n = n0 + wn * WN + 32 * j + n32;
    if (n >= a.n) continue;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int m = m0 + wm * WM + 32 * i + 8 * (e >> 2) + 4 * u + (e & 3);
        if (m < a.m) y[(int64_t)m * a.ldy + n] = acc[i][j][e] * a.alpha;
      }
  }
}

// y = alpha * the sum of the parts (f32, part after part).
__global__ __launch_bounds__(256) void linear_parts_kernel(const float* ws, LinArgs a, int parts) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4, total = a.m * a.n;
  if (i >= total) return;
  f32x4 v = *(const f32x4*)(ws + i);
  for (int p = 1; p < parts; ++p) v += *(const f32x4*)(ws + p * total + i);
  // n is a multiple of 4 here, so the four values are one row's
  const int64_t r = total <= UINT32_MAX ? (int64_t)((uint32_t)i / (uint32_t)a.n) : i / a.n;
  *(f32x4*)((float*)a.y + r * a.ldy + (i - r * a.n)) = v * a.alpha;
}

// Parts of k for the split kernel (0: the library's f32 product), by modelled
// times in us: a slice of a 128 x 128 tile takes a CU 1.1, 1.4 when all CUs
// work (the clock drops), tiles x parts run in rounds of 256, parts are summed
// by one more pass; the library reaches about 120 TFLOP/s on the f32 unit.
// The new form has to win by 5 %.  Measured, library -> this (m x n x k, the
// same operands again and again; over changing ones both take 2-5 % longer):
//   912 x 4096 x 2048 119 -> 89 us, 912 x 12288 x 2048 351 -> 258,
//   912 x 2048 x 6144 174 -> 134 (two parts), 512 x 2048 x 2048 38 -> 34,
//   2048 x 4096 x 2048 235 -> 176, 2048 x 2048 x 6144 342 -> 255;
//   200 x 4096 x 2048 (64 tiles) 39 against 72 stays with the library.
int split_parts(const LinArgs& a, size_t ws_bytes) {
  constexpr int kCus = 256;
  const int64_t tiles = ((a.m + kSplitTile - 1) / kSplitTile) * ((a.n + kSplitTile - 1) / kSplitTile);
  if (a.m < kSplitTile || tiles > (1 << 24)) return 0;
  const double slices = std::ceil((double)a.k / kSliceK);
  double best = 0.95 * (8.0 + 2.0 * (double)a.m * (double)a.n * (double)a.k / 120e6);
  int parts = 0;
  for (int p = 1; p <= 4; p *= 2) {
    const size_t bytes = (size_t)p * a.m * a.n * 4;
    if (p > 1 && (bytes > ws_bytes || a.n % 4 != 0 || slices < 16 * p)) break;
    const int64_t wgs = tiles * p;
    double us = 6.0 + std::ceil(slices / p) * ((double)(wgs / kCus) * 1.4 + (wgs % kCus ? 1.1 : 0.0));
    if (p > 1) us += 4.0 + (double)(bytes + a.m * a.n * 4) / 4e6;
    if (us < best) {
      best = us;
      parts = p;
    }
  }
  return parts;
}

int32_t launch_split(const LinArgs& a, int parts, void* ws, hipStream_t s) {
  const int64_t grid = ((a.m + kSplitTile - 1) / kSplitTile) * ((a.n + kSplitTile - 1) / kSplitTile) * parts;
  LinArgs b = a;
  if (parts > 1) {
    b.y = ws;
    b.ldy = a.n;
    b.alpha = 1.0f;
  }
  hipLaunchKernelGGL(linear_split_kernel, dim3((unsigned)grid), dim3(kSplitWaves * 64), 0, s, b, parts);
  if (parts > 1)
    hipLaunchKernelGGL(linear_parts_kernel, dim3((unsigned)((a.m * a.n / 4 + 255) / 256)), dim3(256), 0, s, (const float*)ws, a, parts);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return cev_fail(CEV_ERR_HIP, "cev_linear launch: %s", hipGetErrorString(e));
  return CEV_OK;
}

struct GatherArgs {
  const void* table;
  const int32_t* ids;
  void* out;
  int64_t n, width, ld_table, table_rows, ld_out;
};

// One thread per element: out[i][e] = table[ids[i]][e] in the output dtype;
// an index outside the table gives a NaN row instead of a stray read.
template <typename T, typename TO>
__global__ __launch_bounds__(256) void gather_rows_kernel(GatherArgs a) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= a.n * a.width) return;
  const int64_t i = idx / a.width, e = idx % a.width;
  const int64_t r = a.ids ? (int64_t)a.ids[i] : i;
  const float v = (r >= 0 && r < a.table_rows) ? to_f32<T>(((const T*)a.table)[r * a.ld_table + e]) : __builtin_nanf("");
  ((TO*)a.out)[i * a.ld_out + e] = from_f32<TO>(v);
}

// The same with one thread per 16 bytes of a table row (rows of both sides
// 16-byte aligned, checked by the launcher).  An element a thread, with a
// 64-bit division each, took 22 us for 3584 rows of 2048 bf16 values, four
// times what their bytes need; this form 11 (rows scattered over the table).
template <typename T, typename TO>
__global__ __launch_bounds__(256) void gather_rows_vec_kernel(GatherArgs a) {
  constexpr int VEC = 16 / (int)sizeof(T);
  const uint32_t nv = (uint32_t)(a.width / VEC), idx = blockIdx.x * 256 + threadIdx.x;
  const uint32_t i = idx / nv, e = (idx - i * nv) * VEC;
  if (i >= a.n) return;
  const int64_t r = a.ids ? (int64_t)a.ids[i] : i;
  const bool ok = r >= 0 && r < a.table_rows;
  const uint4 v = *(const uint4*)((const T*)a.table + (ok ? r : 0) * a.ld_table + e);
  TO out[VEC];
#pragma unroll
  for (int j = 0; j < VEC; ++j) out[j] = from_f32<TO>(ok ? to_f32<T>(((const T*)&v)[j]) : __builtin_nanf(""));
  TO* o = (TO*)a.out + (int64_t)i * a.ld_out + e;
#pragma unroll
  for (int j = 0; j < (int)sizeof out / 16; ++j) ((uint4*)o)[j] = ((const uint4*)out)[j];
  if constexpr (sizeof out < 16) *(uint2*)o = *(const uint2*)out;
}

// hipBLASLt state of one cev_blas handle: the library handle and, per
// problem shape, the matmul descriptor, layouts and the heuristic's algo.
// al256: x, w and y all 256-byte aligned (the alignment the picks below
// were measured at); part of the key, so a plan is never reused on less
// aligned operands than it was made for.
struct GemmKey {
  int dtype, out_dtype;
  int64_t m, n, k, ldx, ldw, ldy;
  size_t ws;
  bool al256;
  bool operator<(const GemmKey& o) const {
    return std::tie(dtype, out_dtype, m, n, k, ldx, ldw, ldy, ws, al256) <
           std::tie(o.dtype, o.out_dtype, o.m, o.n, o.k, o.ldx, o.ldw, o.ldy, o.ws, o.al256);
  }
};
struct GemmPlan {
  hipblasLtMatmulDesc_t desc = nullptr;
  hipblasLtMatrixLayout_t la = nullptr, lb = nullptr, lc = nullptr;
  hipblasLtMatmulAlgo_t algo;
  size_t ws = 0;
};

// Per-shape algorithm picks for bf16 projections of the config-2 pass
// (Qwen3-1.7B: 3584 pass tokens), measured offline with gemm_probe.cpp
// (make gemm-probe): the fastest candidate's hipBLASLt solution index and
// the FNV-1a hash of its kernel name, with the probe's median times of the
// heuristic's first pick and of the pick, in us.  Indices number the
// kernels of one loaded hipBLASLt instance: a pick is used only where its
// index names the same kernel (by hash) in the instance this process
// loaded.  The entries are ROCm 7.2's hipBLASLt (what a host that does not
// load torch binds to); in a torch process libcev_hip.so binds to torch's
// own copy, whose heuristic first picks the probe measured within 2 % of
// its fastest candidate on these shapes, so it has no entries.
// The probe ran every candidate on exactly these shapes and layouts
// (leading dimensions k, k and n, bf16 output, 256-byte aligned operands,
// the 32 MiB workspace); a pick applies to nothing else.  Before use it
// must come back from getAlgosFromIndex, name the recorded kernel and pass
// matmulIsAlgoSupported for the call's layouts with a workspace no larger
// than the caller's; otherwise the heuristic's first pick stays.  The
// library never times candidates itself.
struct GemmPick {
  int64_t m, n, k;
  int index;
  uint64_t name_hash;
};
constexpr GemmPick kPicks[] = {
    {3584, 4096, 2048, 440058, 0x2d1baa9a7bbf205aull},  // q/k/v projection   48.1 -> 45.8
    {3584, 2048, 2048, 440090, 0x1eb4eec7c4241052ull},  // o_proj             34.6 -> 28.0
    {3584, 2048, 6144, 440091, 0x58ff78e43625b963ull},  // down               103.6 -> 74.2
};

uint64_t fnv1a(const std::string& s) {
  uint64_t h = 1469598103934665603ull;
  for (unsigned char c : s) {
    h ^= c;
    h *= 1099511628211ull;
  }
  return h;
}

const GemmPick* find_pick(const GemmKey& key) {
  if (key.dtype != CEV_BF16 || key.out_dtype != CEV_BF16 || !key.al256 || key.ldx != key.k || key.ldw != key.k || key.ldy != key.n)
    return nullptr;
  for (const GemmPick& p : kPicks)
    if (p.m == key.m && p.n == key.n && p.k == key.k) return &p;
  return nullptr;
}
struct Blas {
  hipblasLtHandle_t lt = nullptr;
  std::mutex mu;
  std::map<GemmKey, GemmPlan> plans;
};

hipDataType hip_type(int dtype) { return dtype == CEV_BF16 ? HIP_R_16BF : HIP_R_32F; }

int32_t blas_status(hipblasStatus_t st, const char* what) {
  if (st == HIPBLAS_STATUS_SUCCESS) return CEV_OK;
  return cev_fail(st == HIPBLAS_STATUS_NOT_SUPPORTED ? CEV_ERR_UNSUPPORTED : CEV_ERR_HIP, "cev_linear: %s failed (hipBLAS status %d)", what,
                  (int)st);
}

void destroy_plan(GemmPlan& p) {
  if (p.la) hipblasLtMatrixLayoutDestroy(p.la);
  if (p.lb) hipblasLtMatrixLayoutDestroy(p.lb);
  if (p.lc) hipblasLtMatrixLayoutDestroy(p.lc);
  if (p.desc) hipblasLtMatmulDescDestroy(p.desc);
}

// y (m, n) row-major is y^T (n, m) column-major = w (n, k) . x^T: A = w
// read as a (k, n) column-major matrix, transposed; B = x read as (k, m).
int32_t gemm_plan(Blas& b, const GemmKey& key, GemmPlan** out) {
  auto it = b.plans.find(key);
  if (it != b.plans.end()) {
    *out = &it->second;
    return CEV_OK;
  }
  GemmPlan p;
  int32_t rc = blas_status(hipblasLtMatmulDescCreate(&p.desc, HIPBLAS_COMPUTE_32F, HIP_R_32F), "hipblasLtMatmulDescCreate");
  const hipblasOperation_t ta = HIPBLAS_OP_T, tb = HIPBLAS_OP_N;
  if (!rc) rc = blas_status(hipblasLtMatmulDescSetAttribute(p.desc, HIPBLASLT_MATMUL_DESC_TRANSA, &ta, sizeof ta), "TRANSA");
  if (!rc) rc = blas_status(hipblasLtMatmulDescSetAttribute(p.desc, HIPBLASLT_MATMUL_DESC_TRANSB, &tb, sizeof tb), "TRANSB");
  if (!rc) rc = blas_status(hipblasLtMatrixLayoutCreate(&p.la, hip_type(key.dtype), key.k, key.n, key.ldw), "layout A");
  if (!rc) rc = blas_status(hipblasLtMatrixLayoutCreate(&p.lb, hip_type(key.dtype), key.k, key.m, key.ldx), "layout B");
  if (!rc) rc = blas_status(hipblasLtMatrixLayoutCreate(&p.lc, hip_type(key.out_dtype), key.n, key.m, key.ldy), "layout C");
  hipblasLtMatmulPreference_t pref = nullptr;
  if (!rc) rc = blas_status(hipblasLtMatmulPreferenceCreate(&pref), "preference");
  const uint64_t ws = key.ws;
  if (!rc)
    rc = blas_status(hipblasLtMatmulPreferenceSetAttribute(pref, HIPBLASLT_MATMUL_PREF_MAX_WORKSPACE_BYTES, &ws, sizeof ws), "workspace pref");
  hipblasLtMatmulHeuristicResult_t heur[1];
  int found = 0;
  if (!rc)
    rc = blas_status(hipblasLtMatmulAlgoGetHeuristic(b.lt, p.desc, p.la, p.lb, p.lc, p.lc, pref, 1, heur, &found), "heuristic");
  if (pref) hipblasLtMatmulPreferenceDestroy(pref);
  if (!rc && found < 1) rc = cev_fail(CEV_ERR_UNSUPPORTED, "cev_linear: hipBLASLt has no kernel for this product");
  if (rc) {
    destroy_plan(p);
    return rc;
  }
  p.algo = heur[0].algo;
  p.ws = heur[0].workspaceSize;
  if (const GemmPick* pk = find_pick(key)) {
    std::vector<int> idx{pk->index};
    std::vector<hipblasLtMatmulHeuristicResult_t> res;
    const float one = 1.0f, zero = 0.0f;
    size_t need = 0;
    if (hipblaslt_ext::getAlgosFromIndex(b.lt, idx, res) == HIPBLAS_STATUS_SUCCESS && !res.empty() &&
        fnv1a(hipblaslt_ext::getKernelNameFromAlgo(b.lt, res[0].algo)) == pk->name_hash &&
        hipblaslt_ext::matmulIsAlgoSupported(b.lt, p.desc, &one, p.la, p.lb, &zero, p.lc, p.lc, res[0].algo, need) ==
            HIPBLAS_STATUS_SUCCESS &&
        need <= key.ws) {
      p.algo = res[0].algo;
      p.ws = need;
    }
  }
  *out = &(b.plans[key] = p);
  return CEV_OK;
}

bool aligned256(const void* p) { return ((uintptr_t)p & 255) == 0; }

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

template <typename T>
int32_t launch_rows(const LinArgs& a, int out_dtype, hipStream_t s) {
  const dim3 grid((unsigned)((a.n + kLinWaves - 1) / kLinWaves)), block(kLinWaves * 64);
  // rows held per lane and chunks loaded per batch: fewer rows, deeper batches
  auto go = [&](auto mr_c, auto nb_c) {
    constexpr int MR = decltype(mr_c)::value, NB = decltype(nb_c)::value;
    if (out_dtype == CEV_F32)
      hipLaunchKernelGGL((linear_rows_kernel<T, float, MR, NB>), grid, block, 0, s, a);
    else
      hipLaunchKernelGGL((linear_rows_kernel<T, T, MR, NB>), grid, block, 0, s, a);
  };
  using std::integral_constant;
  if (a.m <= 1)
    go(integral_constant<int, 1>{}, integral_constant<int, 8>{});
  else if (a.m <= 2)
    go(integral_constant<int, 2>{}, integral_constant<int, 8>{});
  else if (a.m <= 4)
    go(integral_constant<int, 4>{}, integral_constant<int, 4>{});
  else
    go(integral_constant<int, kRowsSmall>{}, integral_constant<int, 4>{});
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return cev_fail(CEV_ERR_HIP, "cev_linear launch: %s", hipGetErrorString(e));
  return CEV_OK;
}

}  // namespace

extern "C" int32_t cev_blas_create(cev_blas* handle) {
  CEV_CHECK_ARG(handle != nullptr, "cev_blas_create: null output");
  Blas* b = new Blas;
  int32_t rc = blas_status(hipblasLtCreate(&b->lt), "hipblasLtCreate");
  if (rc) {
    delete b;
    return rc;
  }
  *handle = b;
  return CEV_OK;
}

extern "C" int32_t cev_blas_destroy(cev_blas handle) {
  if (!handle) return CEV_OK;
  Blas* b = (Blas*)handle;
  for (auto& kv : b->plans) destroy_plan(kv.second);
  int32_t rc = blas_status(hipblasLtDestroy(b->lt), "hipblasLtDestroy");
  delete b;
  return rc;
}

extern "C" int32_t cev_linear(cev_blas handle, int32_t dtype, int32_t out_dtype, int64_t m, int64_t n, int64_t k, const void* x, int64_t ldx,
                              const void* w, int64_t ldw, float alpha, void* y, int64_t ldy, void* workspace, size_t workspace_bytes,
                              cev_stream stream) {
  if (dtype != CEV_F32 && dtype != CEV_BF16) return cev_fail(CEV_ERR_UNSUPPORTED, "cev_linear: dtype %d", dtype);
  if (out_dtype != CEV_F32 && out_dtype != dtype)
    return cev_fail(CEV_ERR_UNSUPPORTED, "cev_linear: output dtype %d for input dtype %d", out_dtype, dtype);
  const int vec = dtype == CEV_BF16 ? 8 : 4;
  CEV_CHECK_ARG(m >= 0 && n >= 0 && k >= 0, "cev_linear: negative size");
  CEV_CHECK_ARG(k % vec == 0, "cev_linear: k %lld must be a multiple of %d", (long long)k, vec);
  CEV_CHECK_ARG(std::isfinite(alpha), "cev_linear: alpha must be finite");
  if (m == 0 || n == 0) return CEV_OK;
  CEV_CHECK_ARG(x && w && y, "cev_linear: null buffer");
  CEV_CHECK_ARG(ldx >= k && ldw >= k && ldy >= n && ldx % vec == 0 && ldw % vec == 0, "cev_linear: leading dimensions");
  CEV_CHECK_ARG(aligned16(x) && aligned16(w), "cev_linear: x and w must be 16-byte aligned");
  CEV_CHECK_ARG(n <= INT32_MAX && m <= INT32_MAX && k <= INT32_MAX, "cev_linear: size beyond int32");
  hipStream_t s = (hipStream_t)stream;
  if (k == 0 || m <= kRowsSmall) {
    if (k == 0) CEV_CHECK_ARG(m <= kRowsSmall, "cev_linear: k = 0 supported for at most %d rows", kRowsSmall);
    const int64_t grid = (n + kLinWaves - 1) / kLinWaves;
    if (grid > INT32_MAX) return cev_fail(CEV_ERR_UNSUPPORTED, "cev_linear: n too large");
    LinArgs a{x, w, y, m, n, k, ldx, ldw, ldy, alpha};
    if (dtype == CEV_BF16) return launch_rows<uint16_t>(a, out_dtype, s);
    return launch_rows<float>(a, out_dtype, s);
  }
  // The hipBLASLt algorithm is chosen once per shape and kept, so every
  // operand of that path meets the same alignment (the cached choice never
  // meets a less aligned y than it was chosen for).
  const int ovec = out_dtype == CEV_BF16 ? 8 : 4;
  CEV_CHECK_ARG(aligned16(y) && ldy % ovec == 0, "cev_linear: with more than %d rows y must be 16-byte aligned and ldy a multiple of %d",
                kRowsSmall, ovec);
  CEV_CHECK_ARG(handle != nullptr, "cev_linear: more than %d rows need a cev_blas handle", kRowsSmall);
  CEV_CHECK_ARG(workspace_bytes == 0 || workspace != nullptr, "cev_linear: null workspace of %zu bytes", workspace_bytes);
  if (dtype == CEV_F32) {
    const LinArgs a{x, w, y, m, n, k, ldx, ldw, ldy, alpha};
    const int parts = split_parts(a, aligned16(workspace) ? workspace_bytes : 0);
    if (parts > 0) return launch_split(a, parts, workspace, s);
  }
  Blas* b = (Blas*)handle;
  std::lock_guard<std::mutex> lock(b->mu);
  GemmPlan* p = nullptr;
  const bool al256 = aligned256(x) && aligned256(w) && aligned256(y);
  int32_t rc = gemm_plan(*b, GemmKey{dtype, out_dtype, m, n, k, ldx, ldw, ldy, workspace_bytes, al256}, &p);
  if (rc) return rc;
  const float beta = 0.0f;
  return blas_status(hipblasLtMatmul(b->lt, p->desc, &alpha, w, p->la, x, p->lb, &beta, y, p->lc, y, p->lc, &p->algo, workspace,
                                     workspace_bytes, s),
                     "hipblasLtMatmul");
}

extern "C" int32_t cev_linear_form(int32_t dtype, int64_t m, int64_t n, int64_t k, size_t workspace_bytes, int32_t* form) {
  if (dtype != CEV_F32 && dtype != CEV_BF16) return cev_fail(CEV_ERR_UNSUPPORTED, "cev_linear_form: dtype %d", dtype);
  CEV_CHECK_ARG(form != nullptr && m >= 0 && n >= 0 && k >= 0, "cev_linear_form: null output or negative size");
  LinArgs a{};
  a.m = m, a.n = n, a.k = k;
  const int parts = dtype == CEV_F32 && m > kRowsSmall && n > 0 && k > 0 ? split_parts(a, workspace_bytes) : 0;
  *form = m <= kRowsSmall ? 0 : parts > 0 ? parts : -1;
  return CEV_OK;
}

extern "C" int32_t cev_gather_rows(int32_t dtype, int32_t out_dtype, int64_t n, int64_t width, const void* table, int64_t ld_table,
                                   int64_t table_rows, const int32_t* ids, void* out, int64_t ld_out, cev_stream stream) {
  if (dtype != CEV_F32 && dtype != CEV_BF16) return cev_fail(CEV_ERR_UNSUPPORTED, "cev_gather_rows: dtype %d", dtype);
  if (out_dtype != CEV_F32 && out_dtype != CEV_BF16) return cev_fail(CEV_ERR_UNSUPPORTED, "cev_gather_rows: output dtype %d", out_dtype);
  CEV_CHECK_ARG(n >= 0 && width >= 0 && table_rows >= 0, "cev_gather_rows: negative size");
  if (n == 0 || width == 0) return CEV_OK;
  CEV_CHECK_ARG(table && out, "cev_gather_rows: null buffer");
  CEV_CHECK_ARG(ld_table >= width && ld_out >= width, "cev_gather_rows: leading dimensions");
  CEV_CHECK_ARG(ids || n <= table_rows, "cev_gather_rows: %lld rows from a %lld-row table without ids", (long long)n,
                (long long)table_rows);
  const int64_t grid = (n * width + 255) / 256;
  if (grid > INT32_MAX) return cev_fail(CEV_ERR_UNSUPPORTED, "cev_gather_rows: too many elements");
  GatherArgs a{table, ids, out, n, width, ld_table, table_rows, ld_out};
  hipStream_t s = (hipStream_t)stream;
  const dim3 blk(256);
  const int64_t vec = dtype == CEV_BF16 ? 8 : 4, vecs = n * (width / vec);
  const int64_t osz = out_dtype == CEV_BF16 ? 2 : 4, in_sz = dtype == CEV_BF16 ? 2 : 4;
  const int64_t out_piece = vec * osz < 16 ? vec * osz : 16;  // bytes of one store
  // (an empty table has no row to read in place of a wrong index)
  const bool wide = width % vec == 0 && table_rows > 0 && aligned16(table) && ld_table * in_sz % 16 == 0 && ((uintptr_t)out % out_piece) == 0 &&
                    ld_out * osz % out_piece == 0 && vecs + 255 <= UINT32_MAX;
  const dim3 g((unsigned)(wide ? (vecs + 255) / 256 : grid));
  auto go = [&](auto t_c, auto to_c) {
    using T = decltype(t_c);
    using TO = decltype(to_c);
    if (wide)
      hipLaunchKernelGGL((gather_rows_vec_kernel<T, TO>), g, blk, 0, s, a);
    else
      hipLaunchKernelGGL((gather_rows_kernel<T, TO>), g, blk, 0, s, a);
  };
  if (dtype == CEV_BF16 && out_dtype == CEV_BF16)
    go(uint16_t{}, uint16_t{});
  else if (dtype == CEV_BF16)
    go(uint16_t{}, float{});
  else if (out_dtype == CEV_BF16)
    go(float{}, uint16_t{});
  else
    go(float{}, float{});
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return cev_fail(CEV_ERR_HIP, "cev_gather_rows launch: %s", hipGetErrorString(e));
  return CEV_OK;
}
