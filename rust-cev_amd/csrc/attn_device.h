// What the attention kernels share (packed_attn.hip: 256 query slots a
// workgroup and the merge; fan_attn.hip: 32 slots a workgroup): the launch
// arguments, the plan check, MFMA fragments, K/V sources, the output and the
// split records.
#pragma once
#include <type_traits>

#include "cev_device.h"
#include "cev_internal.h"
#include "cev_plan.h"

struct AttnArgs {
  const void* q;
  const void* kc;
  const void* vc;
  const void* kn;
  const void* vn;
  const void* gate;
  void* out;
  char* ws;  // split records: outputs, then (m, l) pairs (cev_plan.h)
  const int32_t* plan;
  int64_t q_st, q_sh, kc_ss, kc_sh, vc_ss, vc_sh, kn_st, kn_sh, vn_st, vn_sh, g_st, g_sh, o_st, o_sh;
  int32_t n_tiles, t, s_cache, hq, hkv, g, has_gate, n_splits, tile_rows;
  int32_t rows_dense;  // the host plan's tiles cover rows [0, t) in order, each row once
  float scale_log2;
  uint32_t plan_sig;  // signature of the host plan this launch was validated with
  int32_t fan_parts, fan_subs;  // attn_kernel_fan: parts of the key stream (0: not this form), 32-slot groups per tile
};

// The small-launch kernel (fan_attn.hip) of a validated call, without the
// merge of its parts.  It has a code object of its own: with it beside the
// 256-slot kernels, the same instructions of those lay elsewhere against the
// other kernels of a pass in the instruction cache, and one 16-token question
// over a 32k prefix took 42.5 us a pass, 42.2 without it.
int32_t cev_attn_fan_launch(const AttnArgs& a, int32_t dtype, int32_t head_dim, hipStream_t stream);

namespace {

constexpr float kRescale = 8.0f;
// Largest sum of a lane's 16 probabilities of one sub-tile that the d = 128
// loop accepts before it moves the row's max (so p < 2^16 there).
constexpr float kMaxP = 65536.0f;
constexpr float kLog2MaxP = 16.0f;  // log2(kMaxP)

// The plan header on the device must be the host plan's (same signature,
// same launch shape).  A device plan that is not a copy of the validated
// host plan is never followed: the attention kernels fill the whole output
// with NaN instead (poison_output) and the merge pass writes nothing, so a
// stale device plan shows in the result rather than leaving rows unwritten.
// The header is read at once and every field compared (no short-circuit,
// which would make each field a dependent load).
// The header stays in h for the offsets the kernel reads next.
__device__ __forceinline__ bool header_ok(const AttnArgs& a, const cev_plan_header& h) {
  // the section offsets follow the header in order (this also loads them
  // with the other fields)
  constexpr int32_t kHeaderWords = (int32_t)(sizeof(cev_plan_header) / 4);
  return (h.magic == CEV_PLAN_MAGIC) & ((uint32_t)h.sig == a.plan_sig) & (h.n_tiles == a.n_tiles) & (h.t == a.t) &
         (h.s_cache == a.s_cache) & (h.n_splits == a.n_splits) & (h.tiles_off >= kHeaderWords) & (h.segs_off >= h.tiles_off) &
         (h.rows_off >= h.segs_off);
}
__device__ __forceinline__ bool plan_ok(const AttnArgs& a, cev_plan_header& h) {
  h = *(const cev_plan_header*)a.plan;
  return header_ok(a, h);
}

// Workgroup b of the grid writes NaN over output rows [b t / G, (b+1) t / G)
// of every query head (the launcher validated the output strides).
template <typename T, int D>
__device__ void poison_output(const AttnArgs& a) {
  const int64_t G = gridDim.x;
  const int64_t r0 = (int64_t)blockIdx.x * a.t / G, r1 = (int64_t)(blockIdx.x + 1) * a.t / G;
  const int64_t per_row = (int64_t)a.hq * D;
  for (int64_t i = threadIdx.x; i < (r1 - r0) * per_row; i += blockDim.x) {
    const int64_t r = r0 + i / per_row, h = (i % per_row) / D, e = i % D;
    ((T*)a.out)[r * a.o_st + h * a.o_sh + e] = (T)__builtin_nanf("");
  }
}

// Clamps a segment to the key buffer it starts in.
__device__ __forceinline__ int4 clamp_seg(int4 sg, int s_cache, int t) {
  sg.x = max(sg.x, 0);
  const int lim = sg.x < s_cache ? s_cache : s_cache + t;
  sg.y = min(sg.y, lim);
  return sg;
}

__device__ __forceinline__ float gate_value(float o, float g, bool bf16) {
  // out * sigmoid(g), each op in the model dtype (qwen35.rs:556-558)
  if (bf16) {
    float e = bf16_round(expf(-g));
    float den = bf16_round(e + 1.0f);
    // bf16(1 / den) from the hardware reciprocal (1 ulp): den = D 2^p with
    // D an 8-bit integer, a bf16 rounding midpoint is M 2^q with M an odd
    // 9-bit integer, and D M is never a power of two, so 1 / den lies at
    // least 2^-17 (relative) from every midpoint and a 2^-23 error cannot
    // change its bf16 rounding.  Below 2^-126 (den > 2^126) the reciprocal
    // is an f32 denormal, which the division still gives exactly.
    float sg = bf16_round(den < 0x1p126f ? __builtin_amdgcn_rcpf(den) : 1.0f / den);
    return bf16_round(bf16_round(o) * sg);
  }
  return o * (1.0f / (expf(-g) + 1.0f));
}

__device__ __forceinline__ float pair_max(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

__device__ __forceinline__ float pair_sum(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// The larger of x and its value in lane ^ 16 (within each 32-lane half).
__device__ __forceinline__ float pair16_max(float x) {
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// x plus its value in lane ^ 16 (within each 32-lane half).
__device__ __forceinline__ float pair16_sum(float x) {
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

typedef short s16x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ bf16x4 lds_read_tr(const __bf16* p) {
  s16x4 r = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(p));
  return __builtin_bit_cast(bf16x4, r);
}

// --------------------------------------------------------------------------
// Per-dtype MFMA fragments.
//
// bf16 (v_mfma_f32_32x32x16_bf16): Q as the B operand, 8 head-dim values per
// lane per step; P converted to bf16 B operands whose K slot 8u + j of half
// h is S^T register 8h + j (key 16h + 8(j/4) + 4u + j%4 of a sub-tile); the
// V^T A operand comes from ds_read_b64_tr_b16 on the key-major V tile.
//
// f32 (v_mfma_f32_32x32x2_f32, full f32 products): the head-dim order of
// the QK^T K slots is permuted (d = 8k + 4u + r) so a lane reads 4
// consecutive floats for 4 steps; one K=2 PV step per S^T register.
//
// Both expose the work as small steps so the main loop can interleave the
// MFMAs of one sub-tile with the VALU work of another:
//   qk_step(st), st < NQK   - builds one 32x32 S^T sub-tile;
//   pv_step(j),  j < NPV    - adds one sub-tile's V^T . P^T to O;
//   make_p                  - probabilities -> PV operand, plus their sum.
template <typename T, int D>
struct Frag;

#ifndef CEV_VPAD_BF16
#define CEV_VPAD_BF16 32
#endif

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

template <int D>
struct Frag<__bf16, D> {
  static constexpr int BN = D == 128 ? 64 : 32;
  static constexpr int PAD = 8;
  static constexpr int VPAD = CEV_VPAD_BF16;
  static constexpr int VEC = 8;
  static constexpr int NQK = D / 16;
  static constexpr int NPV = 2 * (D / 32);
  typedef bf16x8 Vec;
  struct P {
    bf16x8 h[2];
  };
  bf16x8 q[D / 16];

  __device__ __forceinline__ void load_q(const __bf16* qp, bool ok, int u) {
#pragma unroll
    for (int s = 0; s < D / 16; ++s) {
      bf16x8 z = {};
      q[s] = ok ? *(const bf16x8*)(qp + 16 * s + 8 * u) : z;
    }
  }
  // q * c rounded to bf16: the QK^T MFMAs then give scores already in the
  // base-2 units of the softmax (c = scale * log2 e).
  __device__ __forceinline__ void scale_q(float c) {
#pragma unroll
    for (int s = 0; s < D / 16; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e) q[s][e] = (__bf16)((float)q[s][e] * c);
  }

  // K operand of QK step st: key kt*32 + n, head-dim values 16st + 8u ..
  template <int RS>
  __device__ __forceinline__ static bf16x8 k_frag(const __bf16* sK, int kt, int st, int n, int u) {
    return *(const bf16x8*)&sK[(kt * 32 + n) * RS + 16 * st + 8 * u];
  }
  __device__ __forceinline__ void qk_mfma(const bf16x8& af, int st, f32x16& s) const {
    s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af, q[st], s, 0, 0, 0);
  }
  template <int RS>
  __device__ __forceinline__ void qk_step(const __bf16* sK, int kt, int st, int n, int u, f32x16& s) const {
    qk_mfma(k_frag<RS>(sK, kt, st, n, u), st, s);
  }

  // The row sum is taken over the bf16 probabilities PV multiplies, on the
  // dot-product unit (two products per instruction).
  __device__ __forceinline__ static void make_p(const f32x16& e, P& p, float& rs) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < 8; ++j) p.h[h][j] = (__bf16)e[8 * h + j];
    const bf16x2 one = {(__bf16)1.0f, (__bf16)1.0f};
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < 8; j += 2) rs = __builtin_amdgcn_fdot2_f32_bf16(bf16x2{p.h[h][j], p.h[h][j + 1]}, one, rs, false);
  }

  // Step j = h * (D/32) + dt: o[dt] += V^T(keys of half h) . P^T(half h).
  // Lane (group g16 = lane/16, i = lane%16) reads row kb + i/4, columns
  // d0 + 4(i%4) .. +3; the transpose load hands it 4 consecutive keys of
  // head-dim column d0 + i.
  template <int RS>
  __device__ __forceinline__ static bf16x8 v_frag(const __bf16* sV, int kt, int j, int lane, int u) {
    const int h = j / (D / 32), dt = j % (D / 32);
    const int tr_row = (lane & 15) >> 2;
    const int tr_col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
    const __bf16* vp = sV + (kt * 32 + 16 * h + 4 * u + tr_row) * RS + dt * 32 + tr_col;
    const bf16x4 lo = lds_read_tr(vp);
    const bf16x4 hi = lds_read_tr(vp + 8 * RS);
    return bf16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  }
  __device__ __forceinline__ static void pv_mfma(const bf16x8& af, int j, const P& p, f32x16* o) {
    const int h = j / (D / 32), dt = j % (D / 32);
    o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af, p.h[h], o[dt], 0, 0, 0);
  }
  template <int RS>
  __device__ __forceinline__ void pv_step(const __bf16* sV, int kt, int j, int lane, int u, const P& p, f32x16* o) const {
    pv_mfma(v_frag<RS>(sV, kt, j, lane, u), j, p, o);
  }
};

template <int D>
struct Frag<float, D> {
  static constexpr int BN = 32;
  static constexpr int PAD = 4;
  static constexpr int VPAD = 4;
  static constexpr int VEC = 4;
  static constexpr int NQK = D / 8;
  static constexpr int NPV = 16;
  typedef f32x4 Vec;
  struct P {
    f32x16 v;
  };
  f32x4 q[D / 8];

  __device__ __forceinline__ void load_q(const float* qp, bool ok, int u) {
#pragma unroll
    for (int k = 0; k < D / 8; ++k) q[k] = ok ? *(const f32x4*)(qp + 8 * k + 4 * u) : f32x4{};
  }

  template <int RS>
  __device__ __forceinline__ void qk_step(const float* sK, int kt, int k, int n, int u, f32x16& s) const {
    const f32x4 af = *(const f32x4*)&sK[(kt * 32 + n) * RS + 8 * k + 4 * u];
#pragma unroll
    for (int r = 0; r < 4; ++r) s = __builtin_amdgcn_mfma_f32_32x32x2f32(af[r], q[k][r], s, 0, 0, 0);
  }

  __device__ __forceinline__ static void make_p(const f32x16& e, P& p, float& rs) {
    p.v = e;
#pragma unroll
    for (int i = 0; i < 16; ++i) rs += e[i];
  }

  template <int RS>
  __device__ __forceinline__ void pv_step(const float* sV, int kt, int i, int lane, int u, const P& p, f32x16* o) const {
    const int n = lane & 31;
    const int key = kt * 32 + 8 * (i >> 2) + 4 * u + (i & 3);
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt) o[dt] = __builtin_amdgcn_mfma_f32_32x32x2f32(sV[key * RS + dt * 32 + n], p.v[i], o[dt], 0, 0, 0);
  }
};

template <typename T>
__device__ __forceinline__ void store_vec4(T* p, const float* v);
template <>
__device__ __forceinline__ void store_vec4<__bf16>(__bf16* p, const float* v) {
  bf16x4 r = {(__bf16)v[0], (__bf16)v[1], (__bf16)v[2], (__bf16)v[3]};
  *(bf16x4*)p = r;
}
template <>
__device__ __forceinline__ void store_vec4<float>(float* p, const float* v) {
  *(f32x4*)p = f32x4{v[0], v[1], v[2], v[3]};
}

template <typename T>
__device__ __forceinline__ void load_vec4(const T* p, float* v);
template <>
__device__ __forceinline__ void load_vec4<__bf16>(const __bf16* p, float* v) {
  const bf16x4 g = *(const bf16x4*)p;
  for (int e = 0; e < 4; ++e) v[e] = (float)g[e];
}
template <>
__device__ __forceinline__ void load_vec4<float>(const float* p, float* v) {
  const f32x4 g = *(const f32x4*)p;
  for (int e = 0; e < 4; ++e) v[e] = g[e];
}

// Four values of a record's output as loaded (bf16x4 or f32x4) and their
// f32 form.
template <typename T>
using VecOf = typename std::conditional<sizeof(T) == 2, bf16x4, f32x4>::type;
// E values of T as one load or store: bf16x8 for E = 8, else VecOf<T>.
template <typename T, int E>
using VecN = typename std::conditional<E == 8, bf16x8, VecOf<T>>::type;
__device__ __forceinline__ f32x4 to_f32x4(const bf16x4& v) { return f32x4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]}; }
__device__ __forceinline__ f32x4 to_f32x4(const f32x4& v) { return v; }

// The normalised, optionally gated output of one query slot (row, head):
// lane half ue holds columns 32 dt + 8 q4 + 4 ue .. +3 of o[dt].  bf16
// layers multiply by 1/l (the result is rounded to bf16), f32 layers divide
// by l.  The gate's loads are all issued before the first store, so each of
// the row's output lines is written in one burst; with one load round trip
// between stores, lines sat half written in L2 and went to HBM twice.
template <typename T, int D>
__device__ __forceinline__ void store_output(const AttnArgs& a, int row, int head, int ue, const f32x16* o, float l) {
  constexpr int NDT = D / 32;
  constexpr bool BF = sizeof(T) == 2;
  const float inv = l > 0.0f ? 1.0f / l : 0.0f;
  T* op = (T*)a.out + (int64_t)row * a.o_st + (int64_t)head * a.o_sh;
  auto value = [&](int dt, int i) { return BF ? o[dt][i] * inv : (l > 0.0f ? o[dt][i] / l : 0.0f); };
  if (a.has_gate) {
    const T* gp = (const T*)a.gate + (int64_t)row * a.g_st + (int64_t)head * a.g_sh;
    VecOf<T> graw[NDT][4];
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) graw[dt][q4] = *(const VecOf<T>*)(gp + dt * 32 + 8 * q4 + 4 * ue);
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const f32x4 gv = to_f32x4(graw[dt][q4]);
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = gate_value(value(dt, 4 * q4 + e), gv[e], BF);
        store_vec4<T>(op + dt * 32 + 8 * q4 + 4 * ue, v);
      }
  } else {
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = value(dt, 4 * q4 + e);
        store_vec4<T>(op + dt * 32 + 8 * q4 + 4 * ue, v);
      }
  }
}

// Index of record (row, head, part) in the split workspace.
__device__ __forceinline__ int64_t record_index(const AttnArgs& a, int row, int head, int part) {
  return ((int64_t)row * a.hq + head) * a.n_splits + part;
}
// Output of record i, and the (m, l) region that follows all outputs.
template <typename T, int D>
__device__ __forceinline__ T* record_out(const AttnArgs& a, int64_t i) {
  return (T*)a.ws + i * D;
}
template <typename T, int D>
__device__ __forceinline__ float2* record_ml(const AttnArgs& a) {
  return (float2*)(a.ws + (int64_t)a.t * a.hq * a.n_splits * D * (int64_t)sizeof(T));
}

// Writes this lane's share of partial record (row, head, part): output
// values d .. d+3 of every (dt, q4) slice (d = 32 dt + 8 q4 + 4u), then m
// and l from the lane with u == 0.
template <typename T, int D>
__device__ __forceinline__ void write_record(const AttnArgs& a, int row, int head, int part, const f32x16* o, int u, float m, float l) {
  const int64_t i = record_index(a, row, head, part);
  T* rec = record_out<T, D>(a, i);
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      const int d = dt * 32 + 8 * q4 + 4 * u;
      const float v[4] = {o[dt][4 * q4], o[dt][4 * q4 + 1], o[dt][4 * q4 + 2], o[dt][4 * q4 + 3]};
      store_vec4<T>(rec + d, v);
    }
  if (u == 0) record_ml<T, D>(a)[i] = make_float2(m, l);
}

// Word 3 of a raw buffer resource on gfx9: 32-bit data format, no swizzle.
constexpr int kBufferWord3 = 0x00020000;

// Values the compiler cannot prove wave-uniform (they come through vector
// loads of the plan) but are: readfirstlane moves them to SGPRs, where a
// buffer resource must live.
__device__ __forceinline__ int uniform_i32(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ uint64_t uniform_u64(uint64_t x) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)x);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(x >> 32));
  return ((uint64_t)hi << 32) | lo;
}

// Keeps a value computed where it stands: sched_barrier only fences the
// machine scheduler, and without a use the IR passes sink the row max and
// row sum past the MFMAs they are meant to overlap.
__device__ __forceinline__ void pin(float& x) { asm volatile("" : "+v"(x)); }

// One BN-key chunk of a tile's key stream: keys key0 .. key0 + BN, the first
// nvalid of them inside the segment; local != 0 when the segment's keys are
// masked per row.
struct Chunk {
  int key0, nvalid, local;
};

// Cursor over the BN-key chunks of a tile's segments.  The current segment,
// clamped, stays in SGPRs; the plan is read only when the cursor enters a
// new segment (readfirstlane tells the compiler these vector-loaded values
// are wave-uniform).
template <int BN>
struct ChunkCursor {
  const int4* segs;
  int nseg, s_cache, t;
  int si, k0;
  int4 cur;

  __device__ __forceinline__ int4 seg(int i) const {
    const int4 sg = clamp_seg(segs[i], s_cache, t);
    return make_int4(uniform_i32(sg.x), uniform_i32(sg.y), uniform_i32(sg.z), 0);
  }
  // Positions the cursor on chunk c of the tile's stream.
  __device__ __forceinline__ void seek(int c) {
    si = 0;
    k0 = 0;
    cur = make_int4(0, 0, 0, 0);
    for (; si < nseg; ++si) {
      cur = seg(si);
      const int nch = (max(0, cur.y - cur.x) + BN - 1) / BN;
      if (c < nch) {
        k0 = c * BN;
        return;
      }
      c -= nch;
    }
  }
  __device__ __forceinline__ bool valid() const { return si < nseg; }
  __device__ __forceinline__ void next() {
    k0 += BN;
    if (cur.x + k0 < cur.y) return;
    k0 = 0;
    for (++si; si < nseg; ++si) {
      cur = seg(si);
      if (cur.y > cur.x) return;
    }
  }
  __device__ __forceinline__ Chunk here() const {
    Chunk ch{0, 0, 0};
    if (si < nseg) {
      ch.key0 = cur.x + k0;
      ch.nvalid = max(0, min(BN, cur.y - ch.key0));
      ch.local = cur.z;
    }
    return ch;
  }
};

// K/V rows of one KV head (cache rows [0, s_cache), then the new rows),
// fetched with buffer loads whose byte range ends at a chunk's last valid
// key: rows past it read as zero.
template <typename T>
struct KvSource {
  uint64_t kc, vc, kn, vn;         // row 0 of this head
  int kc_rb, vc_rb, kn_rb, vn_rb;  // row strides in bytes
  int s_cache;

  __device__ __forceinline__ void init(const AttnArgs& a, int kvh) {
    kc = (uint64_t)((const T*)a.kc + kvh * a.kc_sh);
    vc = (uint64_t)((const T*)a.vc + kvh * a.vc_sh);
    kn = (uint64_t)((const T*)a.kn + kvh * a.kn_sh);
    vn = (uint64_t)((const T*)a.vn + kvh * a.vn_sh);
    kc_rb = (int)(a.kc_ss * (int64_t)sizeof(T));
    vc_rb = (int)(a.vc_ss * (int64_t)sizeof(T));
    kn_rb = (int)(a.kn_st * (int64_t)sizeof(T));
    vn_rb = (int)(a.vn_st * (int64_t)sizeof(T));
    s_cache = a.s_cache;
  }
  // Buffer resources for chunk ch and the row strides they use.
  __device__ __forceinline__ void rsrc(const Chunk& ch, __amdgpu_buffer_rsrc_t& rk, __amdgpu_buffer_rsrc_t& rv, int& kr, int& vr) const {
    const bool cached = ch.key0 < s_cache;
    kr = uniform_i32(cached ? kc_rb : kn_rb);
    vr = uniform_i32(cached ? vc_rb : vn_rb);
    const int64_t row0 = cached ? ch.key0 : ch.key0 - s_cache;
    const uint64_t kp = uniform_u64((cached ? kc : kn) + (uint64_t)(row0 * kr));
    const uint64_t vp = uniform_u64((cached ? vc : vn) + (uint64_t)(row0 * vr));
    rk = __builtin_amdgcn_make_buffer_rsrc((void*)kp, (short)0, uniform_i32(ch.nvalid * kr), kBufferWord3);
    rv = __builtin_amdgcn_make_buffer_rsrc((void*)vp, (short)0, uniform_i32(ch.nvalid * vr), kBufferWord3);
  }
};

// Loads this thread's share of chunk ch (NLD 16-byte vectors per tensor).
template <typename T, int D, int NLD, int NT, typename Vec>
__device__ __forceinline__ void load_chunk(const KvSource<T>& src, const Chunk& ch, int tid, Vec* kreg, Vec* vreg) {
  constexpr int VEC = 16 / sizeof(T);
  __amdgpu_buffer_rsrc_t rk, rv;
  int kr, vr;
  src.rsrc(ch, rk, rv, kr, vr);
#pragma unroll
  for (int r = 0; r < NLD; ++r) {
    const int v = tid + r * NT;
    const int key = v / (D / VEC), col = (v % (D / VEC)) * VEC;
    kreg[r] = __builtin_bit_cast(Vec, __builtin_amdgcn_raw_buffer_load_b128(rk, key * kr + col * (int)sizeof(T), 0, 0));
    vreg[r] = __builtin_bit_cast(Vec, __builtin_amdgcn_raw_buffer_load_b128(rv, key * vr + col * (int)sizeof(T), 0, 0));
  }
}

// Query slot (wave, n = lane % 32) of a workgroup over tile rows [r0, r0 +
// len) and KV head kvh holds tile row slot / g and query head slot % g: the
// valid rows of a short tile fill the first waves.
struct SlotRow {
  int row, head, u;
  bool ok;
};
__device__ __forceinline__ SlotRow slot_row(int lane, int wave, int kvh, int g, int r0, int len, int t) {
  const int slot = wave * 32 + (lane & 31);
  const int rit = slot / g;
  SlotRow sr;
  sr.ok = rit < len && r0 + rit < t;
  sr.row = sr.ok ? r0 + rit : 0;
  sr.head = kvh * g + slot % g;
  sr.u = lane >> 5;
  return sr;
}

// This lane's id, computed afresh (opaque to common-subexpression elimination).
__device__ __forceinline__ int fresh_lane_id() {
  int l;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
  return l;
}

namespace pipe {
// 16-byte block of V row `row` that block blk is stored at
__device__ __forceinline__ int v_slot(int blk, int row) { return blk ^ ((row & 3) << 2); }

// s_waitcnt vmcnt(N) with the other counters left alone (gfx9 encoding).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

typedef int i32x2 __attribute__((ext_vector_type(2)));

// V^T operand reads.  The compiler places an s_waitcnt vmcnt(0) before
// every ds_read_b64_tr_b16 it emits while an LDS DMA is in flight (it
// cannot tell the buffers apart), which would drain the whole fetch
// pipeline once per sub-tile.  These reads are issued from asm instead;
// buffer reuse is ordered by the explicit vmcnt wait and barrier at the end
// of each iteration, and wait_tr() below makes a fragment's registers
// depend on the reads having returned.
template <int OFF>
__device__ __forceinline__ i32x2 read_tr(int vaddr) {
  static_assert(OFF >= 0 && OFF < 65536, "ds offset field");
  i32x2 r;
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(r) : "v"(vaddr), "i"(OFF) : "memory");
  return r;
}
// LDS returns in order: once at most N LGKM operations are outstanding,
// every LDS read issued before the last N LDS reads has landed (an older
// scalar load still in flight only makes the wait stricter).
template <int N>
__device__ __forceinline__ void wait_tr(i32x2& lo, i32x2& hi) {
  static_assert(N >= 0 && N < 16, "lgkmcnt range");
  asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(lo), "+v"(hi) : "i"(N));
}
}  // namespace pipe

}  // namespace
