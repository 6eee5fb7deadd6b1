// Small packed-attention launches for gfx950: 32 query slots a workgroup, the
// key stream split over its waves.
#include "attn_device.h"

namespace {

// --------------------------------------------------------------------------
// Small launches, every dtype and head dim: a workgroup of kFanWaves waves
// holds 32 query slots and its waves take the 32-key sub-tiles of the key
// stream in turn, then combine their partials through LDS.
//
// The kernels of packed_attn.hip give a workgroup 256 slots.  With few query
// rows that leaves most CUs idle while one CU's four SIMDs issue the softmax,
// mask and (gated) epilogue instructions of all 256 slots, each instruction 4
// cycles a wave: an 8-workgroup launch measured 15 us and a gated d = 256 one
// 40 us with 2 us of MFMA work.  Here a launch has eight times the
// workgroups, a group's masked keys are cut to the ones its own rows see, and
// a wave carries one sub-tile's worth of every phase.  No barrier until the
// combine: K goes to registers, V into this wave's own LDS (bf16, by DMA
// and read back transposed) or registers (f32), one sub-tile ahead.
// K2 with its merge, traced, before -> now:
//   bf16 d = 128: 1 x 19 tokens after 301 keys 15.0 -> 9.5 us, 8 x 61-77
//   after 74 25.5 -> 11.6, 11 x 21-44 after 421 31.4 -> 16.6;
//   bf16 d = 256 gated: 5 rows of 43 40.0 -> 14.7, 4 x 28-40 after 123
//   42.6 -> 16.2;  f32: 5 x 33-43 after 47 31.2 -> 14.2, 12 x 32 after 256
//   29.3 -> 22.1, 30 x 67-87 after 1915 580 -> 390.
// Each group re-reads its keys (through L2), so long streams under many rows
// stay with the 256-slot kernels; choose_fan (cev_host.cpp) draws the line.
namespace fan {
// The smallest x of the 32 lanes of a wave half.
__device__ __forceinline__ int half_min(int x) {
  x = min(x, (int)dpp_u<0xB1>((uint32_t)x));
  x = min(x, (int)dpp_u<0x4E>((uint32_t)x));
  x = min(x, (int)dpp_u<0x141>((uint32_t)x));
  x = min(x, (int)dpp_u<0x140>((uint32_t)x));
  auto r = __builtin_amdgcn_permlane16_swap((uint32_t)x, (uint32_t)x, false, false);
  return min((int)r[0], (int)r[1]);
}

// Cursor over the 32-key sub-tiles of a tile's segments.  Lane l keeps
// segment 64 b + l of the current batch b of 64, with masked segments cut to
// the keys [lo, hi) that some row of this workgroup's slots can see.
struct Cursor {
  const int4* segs;
  int nseg, s_cache, t, lo, hi;
  int4 batch;
  int si, c_base, nch;
  Chunk seg;  // key0 = first key of segment si, nvalid = its keys

  __device__ __forceinline__ void load_batch(int b) {
    const int i = min(64 * b + (int)(threadIdx.x & 63), nseg - 1);
    int4 sg = clamp_seg(segs[i], s_cache, t);
    if (sg.z) {
      sg.x = max(sg.x, lo);
      sg.y = min(sg.y, hi);
    }
    sg.y = max(sg.y, sg.x);
    batch = sg;
  }
  __device__ __forceinline__ void enter() {
    if (si >= nseg) return;
    if (si > 0 && (si & 63) == 0) load_batch(si >> 6);
    const int l = si & 63;
    seg.key0 = __builtin_amdgcn_readlane(batch.x, l);
    seg.nvalid = __builtin_amdgcn_readlane(batch.y, l) - seg.key0;
    seg.local = __builtin_amdgcn_readlane(batch.z, l);
    nch = (seg.nvalid + 31) >> 5;
  }
  __device__ __forceinline__ void start() {
    si = 0;
    c_base = 0;
    nch = 0;
    seg = Chunk{0, 0, 0};
    if (nseg > 0) load_batch(0);
    enter();
  }
  // Sub-tile c (never before the current segment); false past the end.
  __device__ __forceinline__ bool seek(int c, Chunk& ch) {
    while (si < nseg && c >= c_base + nch) {
      c_base += nch;
      ++si;
      enter();
    }
    if (si >= nseg) return false;
    const int k0 = 32 * (c - c_base);
    ch.key0 = seg.key0 + k0;
    ch.nvalid = min(32, seg.nvalid - k0);
    ch.local = seg.local;
    return true;
  }
  __device__ __forceinline__ int total() {
    while (si < nseg) {
      c_base += nch;
      ++si;
      enter();
    }
    return c_base;
  }
};
}  // namespace fan

// f32: a value as the sum of three bf16 parts (round to nearest each; exact),
// and six of the nine part products of two such operands, small ones first
// (of the three dropped ones the two larger are at most 2^-25 of the product
// each, all three 2^-24).  Six 32x32x16 bf16 MFMAs take 192 cycles where the
// f32 unit takes 512 for the same 16 products; splitting the keys and values
// costs their wave about as much again, so a sub-tile round went from 5.2 to
// 4 us (30 x 67-87 rows after 1915 keys 443 -> 390 us).  The error against 64
// bits is smaller (5.1e-7 against 6.0e-7 there; 21 % over 44 calls of 1-22
// blocks after 38-2518 keys, 12-38 % each): an accumulator is rounded 48 times
// a sub-tile instead of 64.
namespace split {
typedef float f32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void parts(const float* x, bf16x8* p) {
#pragma unroll
  for (int e = 0; e < 8; e += 2) {
    f32x2 r = {x[e], x[e + 1]};
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const bf16x2 b = __builtin_convertvector(r, bf16x2);
      p[i][e] = b[0];
      p[i][e + 1] = b[1];
      r = r - __builtin_convertvector(b, f32x2);
    }
  }
}
__device__ __forceinline__ f32x16 mma(const bf16x8* a, const bf16x8* b, f32x16 c) {
#pragma unroll
  for (int o = 2; o >= 0; --o)
#pragma unroll
    for (int i = 0; i <= o; ++i) c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[o - i], c, 0, 0, 0);
  return c;
}
}  // namespace split

template <typename T, int D>
constexpr int kFanMinWaves = sizeof(T) == 2 && D == 128 ? 2 : 1;
template <typename T, int D>
__global__ __launch_bounds__(kFanWaves * 64) __attribute__((amdgpu_waves_per_eu(kFanMinWaves<T, D>))) void attn_kernel_fan(AttnArgs a) {
  constexpr int NW = kFanWaves;
  using F = Frag<T, D>;
  using P = typename F::P;
  constexpr bool BF = sizeof(T) == 2;
  constexpr int NDT = D / 32;
  constexpr int kRB = D * (int)sizeof(T);          // bytes of one key row
  constexpr int RS = D + 4;                        // row stride (floats) of a partial output in LDS
  constexpr int kVBytes = BF ? NW * 2 * 32 * kRB : 0;  // two V sub-tiles per wave
  constexpr int kOBytes = NW * 32 * RS * 4;        // one partial output per wave
  __shared__ __align__(16) char lds[kVBytes > kOBytes ? kVBytes : kOBytes];
  __shared__ float2 ml[NW * 32];

  cev_plan_header ph;
  if (!plan_ok(a, ph)) {
    poison_output<T, D>(a);
    return;
  }
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform_i32(tid >> 6);
  const int n = lane & 31, u = lane >> 5;
  uint32_t item = blockIdx.x / (uint32_t)a.hkv;
  const int kvh = (int)(blockIdx.x - item * (uint32_t)a.hkv);
  int part = 0;
  if (a.fan_parts > 1) {
    part = (int)(item % (uint32_t)a.fan_parts);
    item /= (uint32_t)a.fan_parts;
  }
  const int tile = (int)(item / (uint32_t)a.fan_subs), sub = (int)item - tile * a.fan_subs;
  const int4 td = ((const int4*)(a.plan + ph.tiles_off))[2 * tile];
  const int gs = __builtin_ctz(a.g);  // g is 1, 2, 4 or 8
  const int sub_rows = 32 >> gs;
  const int r0 = td.x + sub * sub_rows, nr = min(sub_rows, td.y - sub * sub_rows);
  if (nr <= 0) return;
  SlotRow sr;
  sr.ok = (n >> gs) < nr && r0 + (n >> gs) < a.t;
  sr.row = sr.ok ? r0 + (n >> gs) : 0;
  sr.head = kvh * a.g + (n & (a.g - 1));

  const T* const qrow = (const T*)a.q + (int64_t)sr.row * a.q_st + (int64_t)sr.head * a.q_sh;
  F fr;                         // bf16
  bf16x8 qp[BF ? 1 : D / 16][3];  // f32: the parts of q[16 st + 8 u ..]
  auto load_q8 = [&](int st, float* x) {
#pragma unroll
    for (int e = 0; e < 8; e += 4) {
      const f32x4 v = sr.ok ? *(const f32x4*)(qrow + 16 * st + 8 * u + e) : f32x4{};
#pragma unroll
      for (int j = 0; j < 4; ++j) x[e + j] = v[j];
    }
  };
  if constexpr (BF) {
    fr.load_q(qrow, sr.ok, u);
  } else {
#pragma unroll
    for (int st = 0; st < D / 16; ++st) {
      float x[8];
      load_q8(st, x);
      split::parts(x, qp[st]);
    }
  }
  int4 rv = ((const int4*)(a.plan + ph.rows_off))[sr.row];
  if (!sr.ok) rv = make_int4(0, 0, -1, 0);
  fan::Cursor cur;
  cur.segs = (const int4*)(a.plan + ph.segs_off) + td.z;
  cur.nseg = uniform_i32(td.w);
  cur.s_cache = a.s_cache;
  cur.t = a.t;
  {
    // the local keys that some row of these slots sees
    int lo = rv.y > rv.x ? rv.x : INT32_MAX, hi = rv.y > rv.x ? rv.y : 0;
    if (rv.z >= 0) {
      lo = min(lo, rv.z);
      hi = max(hi, rv.z + 1);
    }
    cur.lo = uniform_i32(fan::half_min(lo));
    cur.hi = -uniform_i32(fan::half_min(-hi));
  }
  cur.start();
  int c = wave, c_end = INT32_MAX;
  if (a.fan_parts > 1) {
    const int total = cur.total();
    c = (int)((int64_t)part * total / a.fan_parts) + wave;
    c_end = (int)((int64_t)(part + 1) * total / a.fan_parts);
    cur.start();
  }
  KvSource<T> kvs;
  kvs.init(a, kvh);

  f32x16 o[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) o[dt] = f32x16{};
  float m_run = -1e30f, l_run = 0.0f;
  char* const vl = lds + wave * 2 * 32 * kRB;  // bf16: this wave's V sub-tiles
  const int lds_v = (int)(size_t)(const __attribute__((address_space(3))) char*)vl;
  int voff[NDT];
  if constexpr (BF) {
    const int i = lane & 15, rr = i >> 2, blk = 2 * ((lane >> 4) & 1) + ((i & 3) >> 1);
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) voff[dt] = (4 * u + rr) * kRB + (pipe::v_slot(4 * dt + blk, rr) << 4) + 8 * (i & 1);
  }

  // Loads of one sub-tile: K, 16 bytes of key row n per load, into kf; V into
  // LDS buffer `buf` (bf16) or into vf (f32, issued on its own).  A sub-tile
  // past the end has no valid key: its loads read no memory.
  constexpr int kKLoads = kRB / 32, kVLoads = BF ? kRB / 32 : 0;
  f32x4 kf[kKLoads];
  float vf[BF ? 1 : 16][BF ? 1 : NDT];
  __amdgpu_buffer_rsrc_t rk, rvs;
  int kr, vr;
  auto load_k = [&](const Chunk& x, int buf) {
    kvs.rsrc(x, rk, rvs, kr, vr);
#pragma unroll
    for (int i = 0; i < kKLoads; ++i) {
      // bf16: 8 values at 16 i + 8 u; f32: 4 values at 16 (i / 2) + 8 u + 4 (i % 2)
      const int at = BF ? 32 * i + 16 * u : 64 * (i >> 1) + 32 * u + 16 * (i & 1);
      kf[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rk, n * kr + at, 0, 0));
    }
    if constexpr (BF) {
      constexpr int kRows = 1024 / kRB, kBlk = kRB / 16;  // rows of one 1 KB DMA, 16-byte blocks of a row
#pragma unroll
      for (int r = 0; r < kVLoads; ++r) {
        const int vrow = kRows * r + lane / kBlk;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rvs, (__attribute__((address_space(3))) void*)(vl + buf * (32 * kRB) + 1024 * r), 16,
                                                 vrow * vr + (pipe::v_slot(lane % kBlk, vrow) << 4), 0, 0, 0);
      }
    }
  };
  auto load_v = [&]() {
    if constexpr (!BF) {
#pragma unroll
      for (int i = 0; i < 16; ++i)
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
          vf[i][dt] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rvs, (8 * (i >> 2) + 4 * u + (i & 3)) * vr + (dt * 32 + n) * 4, 0, 0));
    }
  };
  auto at = [&](int i, Chunk& x) {
    x = Chunk{0, 0, 0};
    return i < c_end && cur.seek(i, x);
  };

  // f32: an infinite value (or one above bf16's range) has no parts.  A wave
  // that ends with anything non-finite walks its keys again on the f32 unit.
  bool exact = false;
  const int c_first = c;
  Chunk ch, chn;
  bool more;
  int buf;
  for (;;) {
    more = at(c, ch);
    buf = 0;
    load_k(ch, 0);
    load_v();
    while (more) {
      f32x16 s = f32x16{};
#pragma unroll
      for (int st = 0; st < D / 16; ++st) {
        if constexpr (BF) {
          fr.qk_mfma(__builtin_bit_cast(bf16x8, kf[st]), st, s);
        } else {
          float x[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) x[e] = kf[2 * st + (e >> 2)][e & 3];
          if (!exact) {
            bf16x8 kp[3];
            split::parts(x, kp);
            s = split::mma(kp, qp[st], s);
          } else {
            float q[8];
            load_q8(st, q);
#pragma unroll
            for (int e = 0; e < 8; ++e) s = __builtin_amdgcn_mfma_f32_32x32x2f32(x[e], q[e], s, 0, 0, 0);
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      c += NW;
      more = at(c, chn);
      load_k(chn, buf ^ 1);
      __builtin_amdgcn_sched_barrier(0);
      if (ch.local != 0 || ch.nvalid < 32) {
        // Branch-free on purpose (see attn_kernel_seq).
        const bool all_rows = ch.local == 0;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int kk = 8 * (i >> 2) + 4 * u + (i & 3);
          const int key = ch.key0 + kk;
          const bool vis = (kk < ch.nvalid) & (all_rows | ((key >= rv.x) & (key < rv.y)) | (key == rv.z));
          s[i] = vis ? s[i] : -INFINITY;
        }
      }
      float mx = -INFINITY;
#pragma unroll
      for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[i]);
      const float m_cand = pair_max(mx) * a.scale_log2;
      const bool grow = m_cand > m_run + kRescale;
      if (__ballot(grow)) {
        const float m_new = grow ? m_cand : m_run;
        const float alpha = fast_exp2(m_run - m_new);
        m_run = m_new;
        l_run *= alpha;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) o[dt] *= alpha;
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = fast_exp2(__builtin_fmaf(s[i], a.scale_log2, -m_run));
      P p;
      F::make_p(s, p, l_run);
      if constexpr (BF) {
        // This sub-tile's V is in LDS once only the next one's loads are in
        // flight.  The V^T reads go through asm (pipe::read_tr): the compiler
        // would wait for the next sub-tile's DMA before each.
        pipe::wait_vmcnt<kKLoads + kVLoads>();
        asm volatile("" ::: "memory");
        const int va = lds_v + buf * (32 * kRB);
        constexpr int kGrp = 4;
        pipe::i32x2 f[2][kGrp][2];
        auto issue = [&](auto g_c) {
          constexpr int G = decltype(g_c)::value;
          static_for<kGrp>([&](auto e_c) {
            constexpr int E = decltype(e_c)::value, J = G * kGrp + E;
            constexpr int OFF = 16 * (J / NDT) * kRB;
            f[G & 1][E][0] = pipe::read_tr<OFF>(va + voff[J % NDT]);
            f[G & 1][E][1] = pipe::read_tr<OFF + 8 * kRB>(va + voff[J % NDT]);
          });
        };
        issue(std::integral_constant<int, 0>{});
        static_for<F::NPV / kGrp>([&](auto g_c) {
          constexpr int G = decltype(g_c)::value;
          static_for<kGrp>([&](auto e_c) {
            constexpr int E = decltype(e_c)::value;
            pipe::wait_tr<0>(f[G & 1][E][0], f[G & 1][E][1]);
          });
          if constexpr (G + 1 < F::NPV / kGrp) issue(std::integral_constant<int, G + 1>{});
          static_for<kGrp>([&](auto e_c) {
            constexpr int E = decltype(e_c)::value;
            const bf16x4 lo = __builtin_bit_cast(bf16x4, f[G & 1][E][0]), hi = __builtin_bit_cast(bf16x4, f[G & 1][E][1]);
            F::pv_mfma(bf16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]}, G * kGrp + E, p, o);
          });
        });
      } else {
        if (!exact) {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            float x[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = p.v[8 * h + e];
            bf16x8 pp[3];
            split::parts(x, pp);
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt) {
#pragma unroll
              for (int e = 0; e < 8; ++e) x[e] = vf[8 * h + e][dt];
              bf16x8 vp[3];
              split::parts(x, vp);
              o[dt] = split::mma(vp, pp, o[dt]);
            }
          }
        } else {
#pragma unroll
          for (int i = 0; i < 16; ++i)
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt) o[dt] = __builtin_amdgcn_mfma_f32_32x32x2f32(vf[i][dt], p.v[i], o[dt], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        load_v();
      }
      ch = chn;
      buf ^= 1;
    }
    if constexpr (BF) break;
    float t = l_run * 0.0f + m_run * 0.0f;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) t += o[dt][i] * 0.0f;
    if (exact || !__any(!(t == 0.0f))) break;
    exact = true;
    c = c_first;
    cur.start();
    m_run = -1e30f;
    l_run = 0.0f;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) o[dt] = f32x16{};
  }
  // loads past the end still write zeros into LDS: drain them
  if (BF) pipe::wait_vmcnt<0>();

  // ---- combine the waves' partials through LDS
  const float l = pair_sum(l_run);
  if (BF) __syncthreads();  // every wave is done with its V sub-tile
  float* const ob = (float*)lds;
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4)
      *(f32x4*)(ob + (wave * 32 + n) * RS + dt * 32 + 8 * q4 + 4 * u) = f32x4{o[dt][4 * q4], o[dt][4 * q4 + 1], o[dt][4 * q4 + 2], o[dt][4 * q4 + 3]};
  if (u == 0) ml[wave * 32 + n] = make_float2(m_run, l);
  // thread -> (slot, 8-column unit), the units of a slot side by side
  constexpr int TPS = NW * 2, kUnits = D / 8 / TPS;
  static_assert(D % (8 * TPS) == 0, "units split evenly");
  const int slot = tid / TPS, tu = tid % TPS;
  const int row = r0 + (slot >> gs), head = kvh * a.g + (slot & (a.g - 1));
  const bool ok = (slot >> gs) < nr && row < a.t;
  __syncthreads();
  if (!ok) return;
  float M = -INFINITY, L = 0.0f, w[NW];
#pragma unroll
  for (int i = 0; i < NW; ++i) M = fmaxf(M, ml[i * 32 + slot].x);
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    const float2 v = ml[i * 32 + slot];
    w[i] = fast_exp2(v.x - M);
    L += w[i] * v.y;
  }
  const float inv = L > 0.0f ? 1.0f / L : 0.0f;
#pragma unroll 1
  for (int k = 0; k < kUnits; ++k) {
    const int d = 8 * (tu + k * TPS);
    float x[8] = {};
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      const float* pp = ob + (i * 32 + slot) * RS + d;
      const f32x4 x0 = *(const f32x4*)pp, x1 = *(const f32x4*)(pp + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[e] += w[i] * x0[e];
        x[4 + e] += w[i] * x1[e];
      }
    }
    if (a.fan_parts > 1) {
      const int64_t ri = record_index(a, row, head, part);  // fan_parts == n_splits here
      T* rec = record_out<T, D>(a, ri) + d;
      store_vec4<T>(rec, x);
      store_vec4<T>(rec + 4, x + 4);
      if (d == 0) record_ml<T, D>(a)[ri] = make_float2(M, L);
      continue;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = BF ? x[e] * inv : (L > 0.0f ? x[e] / L : 0.0f);
    if (a.has_gate) {
      float gv[8];
      const T* gp = (const T*)a.gate + (int64_t)row * a.g_st + (int64_t)head * a.g_sh + d;
      load_vec4<T>(gp, gv);
      load_vec4<T>(gp + 4, gv + 4);
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = gate_value(x[e], gv[e], BF);
    }
    T* op = (T*)a.out + (int64_t)row * a.o_st + (int64_t)head * a.o_sh + d;
    store_vec4<T>(op, x);
    store_vec4<T>(op + 4, x + 4);
  }
}

template <typename T, int D>
int32_t launch(const AttnArgs& a, hipStream_t stream) {
  const int64_t grid = (int64_t)a.n_tiles * a.fan_subs * a.fan_parts * a.hkv;
  if (grid > INT32_MAX) return cev_fail(CEV_ERR_UNSUPPORTED, "grid of %lld workgroups is too large", (long long)grid);
  hipLaunchKernelGGL((attn_kernel_fan<T, D>), dim3((unsigned)grid), dim3(kFanWaves * 64), 0, stream, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return cev_fail(CEV_ERR_HIP, "packed attention launch: %s", hipGetErrorString(e));
  return CEV_OK;
}

}  // namespace

int32_t cev_attn_fan_launch(const AttnArgs& a, int32_t dtype, int32_t head_dim, hipStream_t stream) {
  if (dtype == CEV_F32) return launch<float, 128>(a, stream);
  return head_dim == 128 ? launch<__bf16, 128>(a, stream) : launch<__bf16, 256>(a, stream);
}
