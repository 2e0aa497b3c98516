// The grouped UPDATE's token products for narrow experts (I, D <= 512), one
// launch instead of two and no fp32 intermediate, and the APPLY's gate/up.
//
// At the shipped expert widths (192 x 192, 384 x 384) the UPDATE's first stage
// multiplies each token by three small matrices and writes six rows of results:
// its products take a quarter of the time its rows take from and to memory.
// The 256-token kernels of grouped_gemm.hip compute w1^T v in a launch of its
// own (an fp32 round trip of I elements per token), pad 192 rows to 256 and,
// one workgroup per CU, leave memory idle in every prologue and epilogue.
// Here a workgroup takes 64 hidden units of one expert and 128 tokens: the
// w1 columns times v, then the w0 and w2 rows times k, all in the same lanes
// (wave w holds tokens 32 w .. + 31 of all 64 units: 96 accumulators), so the
// pointwise part runs in registers, each wave on its own.  A ring of three
// 16 KiB stages (32 k of 128 tokens and of the weights) lets three workgroups
// share a CU, one's epilogue under the others' loads (two in the backward, whose
// pass holds the saved inputs beside the accumulators).
//
// 48 experts of 192 x 192 over 196 608 tokens, bound by the rows' stream:
//   stage 1 with the saves  273 us (two launches) -> 158 (600 MB, 3.8 TB/s)
//   backward's second pass  302 us (two launches) -> 223 (830 MB, 3.7 TB/s)
// 96 of 384 x 384 over 16 384 tokens, without saves: 89 -> 45 us; gate/up 42 ->
// 31, of 48 x 192 x 192 17 -> 10.7 (against apply_kernel's 256 x 128 tiles).
// Stage 1 of every I, D up to 512 measured gains, the backward but for the widest
// of many tokens (narrow_stage1, narrow_bwd); past 512 long segments were not
// timed, and a token tile is read by more than eight unit groups: the 256-token
// tiles' kernels.
#include "narrow.h"
#include "tile192.h"

namespace uttt {
namespace {

using namespace pipe;
using t192::kTK;
using t192::kTThreads;
using t192::Loader;

constexpr int kHid = 64;                 // hidden units per workgroup
constexpr int kTok = 128;                // tokens per workgroup
constexpr int kSlot = 16 * 1024;         // weights (8 KiB; w1 4 KiB) | tokens (8 KiB)
constexpr int kSlotTok = 8 * 1024;
constexpr int kRing = 3;
constexpr int kPlane = 32 * kHid * 2;    // one tensor's rows of a wave's 32 tokens: 4 KiB
constexpr int kWavePlanes = 3;
static_assert(kRing * kSlot >= 4 * kWavePlanes * kPlane, "epilogue planes fit in the ring");

struct NarrowArgs {
  const uint16_t* w02;  // [B, E, 2I, D]
  const uint16_t* w1;   // [B, E, D, I]
  const uint16_t* k;    // [B, N, D]
  const uint16_t* v;    // [B, N, D]
  const int32_t* gs;
  int B, E, I, D, N, m_tiles, n_tiles_ub;
  const int32_t* src;   // gate/up: rows of k [B, T, D] (optional)
  long long src_sb;
  int T;
};

// s_waitcnt lgkmcnt(N) that redefines the fragment registers.
template <int N, int M>
__device__ __forceinline__ void wait_frags(bf16x8 (&a)[M], bf16x8& b) {
  i32x4 rb = __builtin_bit_cast(i32x4, b), r[M];
#pragma unroll
  for (int i = 0; i < M; ++i) r[i] = __builtin_bit_cast(i32x4, a[i]);
  if constexpr (M == 2)
    asm volatile("s_waitcnt lgkmcnt(%3)" : "+v"(r[0]), "+v"(r[1]), "+v"(rb) : "i"(N) : "memory");
  else
    asm volatile("s_waitcnt lgkmcnt(%5)"
                 : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]), "+v"(rb)
                 : "i"(N)
                 : "memory");
#pragma unroll
  for (int i = 0; i < M; ++i) a[i] = __builtin_bit_cast(bf16x8, r[i]);
  b = __builtin_bit_cast(bf16x8, rb);
}

// A wave's place in the epilogue: its tokens and hidden units, and its 12 KiB
// of LDS (three planes of [32 tokens][64 units] bf16 in 16-byte chunks, chunk c
// of token t in slot c ^ ((t >> 1) & 7): the 8-byte accesses of one unit
// quadruple over 32 tokens and the 16-byte accesses along rows both cover the
// banks evenly).
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
struct WaveCtx {
  int b, mt, h0, nv;  // nv: this wave's valid tokens (> 0)
  int64_t row0;       // first token row (b * N + ...)
  uint8_t* lds;

  __device__ __forceinline__ uint32_t quad_at(int i, int q) const {
    const int lane = threadIdx.x & 63, t = lane & 31;
    return (uint32_t)(t * 128 + (((4 * i + q) ^ ((t >> 1) & 7)) << 4) + 8 * (lane >> 5));
  }
  // units 32 i + 8 q + 4 (lane / 32) .. + 3 of this lane's token
  __device__ __forceinline__ void put(int plane, int i, int q, const float (&v)[4]) const {
    *reinterpret_cast<uint2*>(lds + plane * kPlane + quad_at(i, q)) =
        make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
  }
  __device__ __forceinline__ uint2 get(int plane, int i, int q) const {
    return *reinterpret_cast<const uint2*>(lds + plane * kPlane + quad_at(i, q));
  }
  __device__ __forceinline__ int lane_unit(int i, int q) const {
    return h0 + 32 * i + 8 * q + 4 * ((threadIdx.x & 63) >> 5);
  }
  // the LDS accesses of one wave complete in order: only the compiler has to
  // keep them so
  __device__ __forceinline__ static void fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  __device__ __forceinline__ uint32_t row_at(int r, int* tok, int* unit) const {
    const int lane = threadIdx.x & 63;
    *tok = r * 8 + (lane >> 3);
    *unit = 8 * (lane & 7);
    return (uint32_t)(*tok * 128 + (((lane & 7) ^ ((*tok >> 1) & 7)) << 4));
  }
  // a plane to columns col0 + h0 .. of out rows [.., ld], 128 bytes per token
  template <bool NT = false>
  __device__ __forceinline__ void store(int plane, uint16_t* out, int ld, int col0, int I) const {
    uint16_t* o = uniform_ptr(out + row0 * ld + col0 + h0);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      int t, u;
      const uint32_t at = row_at(r, &t, &u);
      const u32x4 x = *reinterpret_cast<const u32x4*>(lds + plane * kPlane + at);
      if (t < nv && h0 + u < I) {
        u32x4* dst = reinterpret_cast<u32x4*>(o + (uint32_t)(t * ld + u));
        if constexpr (NT) __builtin_nontemporal_store(x, dst);
        else *dst = x;
      }
    }
  }
  // columns col0 + h0 .. of in rows, from clamped (always valid) addresses
  __device__ __forceinline__ void fetch(u32x4 (&x)[4], const uint16_t* in, int ld, int col0,
                                        int I) const {
    const uint16_t* o = uniform_ptr(in + row0 * ld + col0 + h0);
    static_for<4>([&](auto R) __attribute__((always_inline)) {
      int t, u;
      row_at(R, &t, &u);
      x[R] = *reinterpret_cast<const u32x4*>(
          o + (uint32_t)(min(t, nv - 1) * ld + (h0 + u < I ? u : 0)));
    });
  }
  __device__ __forceinline__ void stage(int plane, const u32x4 (&x)[4]) const {
    static_for<4>([&](auto R) __attribute__((always_inline)) {
      int t, u;
      const uint32_t at = row_at(R, &t, &u);
      *reinterpret_cast<u32x4*>(lds + plane * kPlane + at) = x[R];
    });
  }
};

__device__ __forceinline__ void quad(const f32x16& a, int q, float (&v)[4]) {
#pragma unroll
  for (int u = 0; u < 4; ++u) v[u] = a[q * 4 + u];
}
__device__ __forceinline__ void unpack4(uint32_t x, uint32_t y, float (&v)[4]) {
  v[0] = bf16_to_f32((uint16_t)(x & 0xffffu));
  v[1] = bf16_to_f32((uint16_t)(x >> 16));
  v[2] = bf16_to_f32((uint16_t)(y & 0xffffu));
  v[3] = bf16_to_f32((uint16_t)(y >> 16));
}

// --- APPLY gate/up (y0 = w0 x, y2 = w2 x)
struct NarrowSwiGLU {
  static constexpr int kWgsPerCu = 3;
  static constexpr bool kThree = false;
  struct Args {
    uint16_t* hid;  // [B, N, I]
  };
  __device__ __forceinline__ static void apply(const Args& ea, const NarrowArgs& a,
                                               const WaveCtx& c, const f32x16 (&)[2],
                                               const f32x16 (&y)[4]) {
    static_for<8>([&](auto Q) __attribute__((always_inline)) {
      constexpr int i = decltype(Q)::value / 4, q = decltype(Q)::value % 4;
      float y0[4], y2[4], h[4];
      quad(y[i], q, y0);
      quad(y[2 + i], q, y2);
#pragma unroll
      for (int u = 0; u < 4; ++u) h[u] = y2[u] * (y0[u] * sigmoidf_(y0[u]));
      c.put(0, i, q, h);
    });
    WaveCtx::fence();
    c.store(0, ea.hid, a.I, 0, a.I);
  }
};

// --- UPDATE stage 1 (dh = w1^T v, y0 = w0 k, y2 = w2 k): as EpiS1 of
// grouped_gemm.hip, the same operations on the same values.
template <class LR>
struct NarrowS1 {
  static constexpr int kWgsPerCu = 3;
  static constexpr bool kThree = true;  // the w1 product too
  using S = typename LR::S;
  struct Args {
    const S *lr0, *lr1, *lr2;           // [B, N] or null (1)
    uint16_t *dy, *hid;                 // [B, N, 2I], [B, N, I]
    uint16_t *y_save, *dh_save;         // optional
  };
  __device__ __forceinline__ static void apply(const Args& ea, const NarrowArgs& a,
                                               const WaveCtx& c, const f32x16 (&dh)[2],
                                               const f32x16 (&y)[4]) {
    const int64_t li = c.row0 + min((int)(threadIdx.x & 31), c.nv - 1);
    float l0 = 1.0f, l1 = 1.0f, l2 = 1.0f;
    if (ea.lr0 != nullptr) {
      l0 = LR::load(ea.lr0[li]);
      l1 = LR::load(ea.lr1[li]);
      l2 = LR::load(ea.lr2[li]);
    }
    const int I = a.I;
    if (ea.y_save != nullptr) {  // the values the backward would recompute, rounded as it does
      static_for<8>([&](auto Q) __attribute__((always_inline)) {
        constexpr int i = decltype(Q)::value / 4, q = decltype(Q)::value % 4;
        float x[4];
        quad(y[i], q, x);
        c.put(0, i, q, x);
        quad(y[2 + i], q, x);
        c.put(1, i, q, x);
        quad(dh[i], q, x);
        c.put(2, i, q, x);
      });
      WaveCtx::fence();
      c.template store<true>(0, ea.y_save, 2 * I, 0, I);
      c.template store<true>(1, ea.y_save, 2 * I, I, I);
      c.template store<true>(2, ea.dh_save, I, 0, I);
      WaveCtx::fence();
    }
    static_for<8>([&](auto Q) __attribute__((always_inline)) {
      constexpr int i = decltype(Q)::value / 4, q = decltype(Q)::value % 4;
      float y0[4], y2[4], d[4], d0[4], d2[4], hh[4];
      quad(y[i], q, y0);
      quad(y[2 + i], q, y2);
      quad(dh[i], q, d);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float sg = sigmoidf_(y0[u]);
        const float sw = sg * y0[u];
        d0[u] = sg * y2[u] * d[u] * (1.0f + y0[u] * (1.0f - sg)) * l0;
        d2[u] = sw * d[u] * l2;
        hh[u] = sw * y2[u] * l1;
      }
      c.put(0, i, q, d0);
      c.put(1, i, q, d2);
      c.put(2, i, q, hh);
    });
    WaveCtx::fence();
    c.store(0, ea.dy, 2 * I, 0, I);
    c.store(1, ea.dy, 2 * I, I, I);
    c.store(2, ea.hid, I, 0, I);
  }
};

// --- UPDATE backward from the saved values (gd = gw1^T v, gy0 | gy2 =
// gw0_w2 k, all three rounded to bf16): as EpiBwdSaved of grouped_gemm.hip,
// with gd from the accumulators.  lr_part[j][mt][b][tok] sums this tile's 64
// units.
template <class LR>
struct NarrowBwd {
  static constexpr int kWgsPerCu = 2;
  static constexpr bool kThree = true;
  using S = typename LR::S;
  struct Args {
    const uint16_t *y_saved, *dh_saved;  // [B, N, 2I], [B, N, I]
    const S *lr0, *lr1, *lr2;
    uint16_t *gdh, *gx, *dx, *hlr;
    float* lr_part;
  };
  __device__ __forceinline__ static void apply(const Args& ea, const NarrowArgs& a,
                                               const WaveCtx& c, const f32x16 (&gd)[2],
                                               const f32x16 (&gy)[4]) {
    const int I = a.I, lane = threadIdx.x & 63, t = lane & 31;
    const int64_t li = c.row0 + min(t, c.nv - 1);
    const S r0 = ea.lr0[li], r1 = ea.lr1[li], r2 = ea.lr2[li];
    {
      u32x4 x0[4], x2[4], xd[4];
      c.fetch(x0, ea.y_saved, 2 * I, 0, I);
      c.fetch(x2, ea.y_saved, 2 * I, I, I);
      c.fetch(xd, ea.dh_saved, I, 0, I);
      c.stage(0, x0);
      c.stage(1, x2);
      c.stage(2, xd);
    }
    const float L0 = LR::load(r0), L1 = LR::load(r1), L2 = LR::load(r2);
    WaveCtx::fence();
    uint32_t p0[16], p2[16], pd[16];  // the inputs, packed
    float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f;
    // the outputs take the place of the inputs that this lane reads
    static_for<8>([&](auto Q) __attribute__((always_inline)) {
      constexpr int i = decltype(Q)::value / 4, q = decltype(Q)::value % 4;
      constexpr int at = 2 * decltype(Q)::value;
      const uint2 in0 = c.get(0, i, q), in2 = c.get(1, i, q), ind = c.get(2, i, q);
      p0[at] = in0.x, p0[at + 1] = in0.y;
      p2[at] = in2.x, p2[at + 1] = in2.y;
      pd[at] = ind.x, pd[at + 1] = ind.y;
      float y0v[4], y2v[4], dh[4], g0[4], g2[4], gd_[4], o_gdh[4], o_gx0[4], o_gx2[4];
      unpack4(p0[at], p0[at + 1], y0v);
      unpack4(p2[at], p2[at + 1], y2v);
      unpack4(pd[at], pd[at + 1], dh);
      quad(gy[i], q, g0);
      quad(gy[2 + i], q, g2);
      quad(gd[i], q, gd_);
      float t0 = 0.0f, t1 = 0.0f, t2 = 0.0f;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float y0 = y0v[u], y2 = y2v[u];
        const float gd0 = bf16r(g0[u]), gd2 = bf16r(g2[u]), gdv = bf16r(gd_[u]);
        const float sg = sigmoidf_(y0);
        const float silu = sg * y0;
        const float mul = sg * (1.0f + y0 * (1.0f - sg));  // silu'(y0)
        const float ds = sg * (1.0f - sg);                  // sigmoid'(y0)
        o_gdh[u] = gd0 * L0 * y2 * mul + gd2 * L2 * silu;
        o_gx2[u] = gd0 * L0 * dh[u] * mul + gdv * L1 * silu;
        const float gsig = gd0 * L0 * dh[u] * y2 * (1.0f + y0 - 2.0f * sg * y0);
        o_gx0[u] = (gd2 * L2 * dh[u] + gdv * L1 * y2) * mul + gd0 * L0 * dh[u] * y2 * ds +
                   gsig * ds;
        t0 += gd0 * dh[u] * y2 * mul;
        t1 += gdv * y2 * silu;
        t2 += gd2 * dh[u] * silu;
      }
      const bool in = c.lane_unit(i, q) < I;  // I is a multiple of 8: all four or none
      s0 += in ? t0 : 0.0f;
      s1 += in ? t1 : 0.0f;
      s2 += in ? t2 : 0.0f;
      c.put(0, i, q, o_gdh);
      c.put(1, i, q, o_gx0);
      c.put(2, i, q, o_gx2);
      // one quadruple's values at a time in registers: the sums are due here
      asm volatile("" : "+v"(s0), "+v"(s1), "+v"(s2));
      __builtin_amdgcn_sched_barrier(0);
    });
    WaveCtx::fence();
    c.store(0, ea.gdh, I, 0, I);
    c.store(1, ea.gx, 2 * I, 0, I);
    c.store(2, ea.gx, 2 * I, I, I);
    s0 += __shfl_xor(s0, 32);
    s1 += __shfl_xor(s1, 32);
    s2 += __shfl_xor(s2, 32);
    if (lane < 32 && t < c.nv) {
      const int64_t plane = (int64_t)a.m_tiles * a.B * a.N;
      const int64_t o = (int64_t)c.mt * a.B * a.N + c.row0 + t;
      ea.lr_part[o] = s0;
      ea.lr_part[plane + o] = s1;
      ea.lr_part[2 * plane + o] = s2;
    }
    WaveCtx::fence();
    static_for<8>([&](auto Q) __attribute__((always_inline)) {
      constexpr int i = decltype(Q)::value / 4, q = decltype(Q)::value % 4;
      float y0v[4], y2v[4], dh[4], o_dx0[4], o_dx2[4], o_hl[4];
      constexpr int at = 2 * decltype(Q)::value;
      // opaque copies: the first pass's values are recomputed, not kept in registers
      asm volatile("" : "+v"(p0[at]), "+v"(p0[at + 1]), "+v"(p2[at]), "+v"(p2[at + 1]),
                        "+v"(pd[at]), "+v"(pd[at + 1]));
      unpack4(p0[at], p0[at + 1], y0v);
      unpack4(p2[at], p2[at + 1], y2v);
      unpack4(pd[at], pd[at + 1], dh);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float y0 = y0v[u], y2 = y2v[u];
        const float sg = sigmoidf_(y0);
        const float silu = sg * y0;
        const float mul = sg * (1.0f + y0 * (1.0f - sg));
        o_dx0[u] = dh[u] * y2 * mul * L0;
        o_dx2[u] = silu * dh[u] * L2;
        o_hl[u] = L1 * y2 * silu;
      }
      c.put(0, i, q, o_dx0);
      c.put(1, i, q, o_dx2);
      c.put(2, i, q, o_hl);
      __builtin_amdgcn_sched_barrier(0);
    });
    WaveCtx::fence();
    c.store(0, ea.dx, 2 * I, 0, I);
    c.store(1, ea.dx, 2 * I, I, I);
    c.store(2, ea.hlr, I, 0, I);
  }
};

// Stage s of one product into a ring slot.
template <class LA, class LT>
__device__ __forceinline__ void issue_stage(LA& la, LT& lt, int s, uint8_t* slot) {
  la.issue(s, slot);
  lt.issue(s, slot + kSlotTok);
}

// One stage (its loads have landed for this wave): barrier, next_issue(), the
// fragments of both k-substeps, the products.
template <class Next>
__device__ __forceinline__ void dh_stage(f32x16 (&dh)[2], const uint8_t* slot, int w,
                                         const uint32_t (&ar)[2], const uint32_t (&ak)[2],
                                         Next&& next_issue) {
  block_barrier();
  __builtin_amdgcn_sched_barrier(0);
  const uint32_t ta = lds_addr(slot), tb = ta + kSlotTok + w * 2048;
  bf16x8 fa[2][2], fb[2];
  static_for<2>([&](auto KS) __attribute__((always_inline)) {
    static_for<2>([&](auto I) __attribute__((always_inline)) {
      const i16x4 x0 = ds_tr16_asm<decltype(KS)::value * 2048>(ta + ar[I]);
      const i16x4 x1 = ds_tr16_asm<decltype(KS)::value * 2048 + 512>(ta + ar[I]);
      fa[KS][I] =
          __builtin_bit_cast(bf16x8, __builtin_shufflevector(x0, x1, 0, 1, 2, 3, 4, 5, 6, 7));
    });
    fb[KS] = ds_b128_asm<0>(tb + ak[KS]);
  });
  next_issue();
  __builtin_amdgcn_sched_barrier(0);
  wait_frags<5>(fa[0], fb[0]);
  static_for<2>([&](auto I) __attribute__((always_inline)) {
    dh[I] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[0][I], fb[0], dh[I], 0, 0, 0);
  });
  __builtin_amdgcn_sched_barrier(0);
  wait_frags<0>(fa[1], fb[1]);
  static_for<2>([&](auto I) __attribute__((always_inline)) {
    dh[I] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[1][I], fb[1], dh[I], 0, 0, 0);
  });
  __builtin_amdgcn_sched_barrier(0);
}
template <class Next>
__device__ __forceinline__ void y_stage(f32x16 (&y)[4], const uint8_t* slot, int w,
                                        const uint32_t (&ak)[2], Next&& next_issue) {
  block_barrier();
  __builtin_amdgcn_sched_barrier(0);
  const uint32_t ta = lds_addr(slot), tb = ta + kSlotTok + w * 2048;
  bf16x8 fa[2][4], fb[2];
  static_for<2>([&](auto KS) __attribute__((always_inline)) {
    static_for<4>([&](auto I) __attribute__((always_inline)) {
      fa[KS][I] = ds_b128_asm<decltype(I)::value * 2048>(ta + ak[KS]);
    });
    fb[KS] = ds_b128_asm<0>(tb + ak[KS]);
  });
  next_issue();
  __builtin_amdgcn_sched_barrier(0);
  wait_frags<5>(fa[0], fb[0]);
  static_for<4>([&](auto I) __attribute__((always_inline)) {
    y[I] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[0][I], fb[0], y[I], 0, 0, 0);
  });
  __builtin_amdgcn_sched_barrier(0);
  wait_frags<0>(fa[1], fb[1]);
  static_for<4>([&](auto I) __attribute__((always_inline)) {
    y[I] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[1][I], fb[1], y[I], 0, 0, 0);
  });
  __builtin_amdgcn_sched_barrier(0);
}

template <class Epi>
__device__ __forceinline__ void narrow_body(const NarrowArgs& a, const typename Epi::Args& ea,
                                            uint8_t* ring) {
  // the m-tiles of one token tile run on one XCD: they read the same token rows
  const int loc = blockIdx.x / kXcds;
  const int unit = loc / a.m_tiles * kXcds + blockIdx.x % kXcds;
  const int mt = loc % a.m_tiles;
  if (unit >= a.B * a.n_tiles_ub) return;
  const int b = unit / a.n_tiles_ub;
  const TokenTile tt =
      find_token_tile<kTok>(a.gs + (int64_t)b * a.E, a.E, a.N, unit - b * a.n_tiles_ub);
  if (tt.e < 0) return;
  const int h0 = mt * kHid;
  const int64_t ge = (int64_t)b * a.E + tt.e;
  const int64_t row = (int64_t)b * a.N + tt.start;

  Loader<RMajor, kHid> l1;        // w1[:, h0 ..]
  Loader<KMajor, 2 * kHid> l02;   // w0[h0 ..] | w2[h0 ..]
  Loader<KMajor, kTok> lv, lk;
  if constexpr (Epi::kThree) {
    l1.init(Operand{a.w1 + ge * a.D * a.I, a.I, a.I, a.D}, h0);
    lv.init(Operand{a.v + row * a.D, a.D, tt.size, a.D}, tt.n0);
  }
  l02.init(Operand{a.w02 + ge * 2 * a.I * a.D, a.D, a.I, a.D}, h0, kHid, a.I * a.D);
  if (!Epi::kThree && a.src != nullptr) {
    const int32_t* src = a.src + (int64_t)b * a.src_sb + tt.start;
    lk.init_gather(a.k + (int64_t)b * a.T * a.D, a.D, a.D, [&](int r) __attribute__((always_inline)) {
      // an index outside [0, T) reads row T - 1
      return (int)min((uint32_t)src[min(tt.n0 + r, tt.size - 1)], (uint32_t)(a.T - 1));
    });
  } else {
    lk.init(Operand{a.k + row * a.D, a.D, tt.size, a.D}, tt.n0);
  }

  const int nk = (a.D + kTK - 1) / kTK;
  uint8_t *p0 = ring, *p1 = ring + kSlot, *p2 = ring + 2 * kSlot;
  auto rotate = [&]() __attribute__((always_inline)) {
    uint8_t* t = p0;
    p0 = p1;
    p1 = p2;
    p2 = t;
  };

  const int lane = threadIdx.x & 63, w = wave_id();
  uint32_t ak[2];  // K-major fragment offsets per k-substep
  {
    const int r = lane & 31;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
      ak[ks] = (uint32_t)((r * 4 + ((2 * ks + (lane >> 5)) ^ ((r >> 2) & 3))) * 16);
  }
  uint32_t ar[2];  // row-major fragment offsets per 32-unit block
  {
    const int g = lane >> 4, s = lane & 15, j = s >> 2, q = s & 3;
    const int k0 = 8 * (g >> 1) + j, x = (j >> 1) & 1;
#pragma unroll
    for (int i = 0; i < 2; ++i)
      ar[i] = (uint32_t)(k0 * 128 + (4 * (i ^ x) + 2 * (g & 1) + (q >> 1)) * 16 + 8 * (q & 1));
  }

  f32x16 dh[2], y[4];
#pragma unroll
  for (int u = 0; u < 16; ++u) {
    dh[0][u] = dh[1][u] = 0.0f;
    y[0][u] = y[1][u] = y[2][u] = y[3][u] = 0.0f;
  }
  // Stages 0 .. nk-1 are the w1 product's, then nk of the w0 | w2 product.  A
  // stage: wait for its loads (the next stage's stay in flight: 3, or 4 for
  // w0 | w2), barrier (it landed for every wave, every wave is done with the
  // slot of the stage before), issue the stage after the next into that slot,
  // read both k-substeps' fragments, multiply.
#define UTTT_DH_STAGE(...) \
  dh_stage(dh, p0, w, ar, ak, [&]() __attribute__((always_inline)) { __VA_ARGS__; }), rotate()
#define UTTT_Y_STAGE(...) \
  y_stage(y, p0, w, ak, [&]() __attribute__((always_inline)) { __VA_ARGS__; }), rotate()
  // D > kTK: at least two stages of each product
  if constexpr (Epi::kThree) {
    issue_stage(l1, lv, 0, p0);
    issue_stage(l1, lv, 1, p1);
    for (int s = 0; s < nk - 2; ++s) {
      wait_vmcnt<3>();
      UTTT_DH_STAGE(issue_stage(l1, lv, s + 2, p2));
    }
    wait_vmcnt<3>();
    UTTT_DH_STAGE(issue_stage(l02, lk, 0, p2));
    wait_vmcnt<4>();
    UTTT_DH_STAGE(issue_stage(l02, lk, 1, p2));
  } else {
    issue_stage(l02, lk, 0, p0);
    issue_stage(l02, lk, 1, p1);
  }
  for (int s = 0; s < nk - 2; ++s) {
    wait_vmcnt<4>();
    UTTT_Y_STAGE(issue_stage(l02, lk, s + 2, p2));
  }
  wait_vmcnt<4>();
  UTTT_Y_STAGE();
  wait_vmcnt<0>();
  UTTT_Y_STAGE();
#undef UTTT_DH_STAGE
#undef UTTT_Y_STAGE
  block_barrier();  // every wave is done reading the ring
  const int n0 = __builtin_amdgcn_readfirstlane(after_loop(tt.n0) + 32 * w);
  const int nv = __builtin_amdgcn_readfirstlane(min(after_loop(tt.size) - n0, 32));
  if (nv <= 0) return;
  const WaveCtx c{b, mt, after_loop(h0), nv, (int64_t)b * a.N + after_loop(tt.start) + n0,
                  ring + w * (kWavePlanes * kPlane)};
  Epi::apply(ea, a, c, dh, y);
}

template <class Epi>
__global__ __launch_bounds__(kTThreads, Epi::kWgsPerCu) void narrow_kernel(NarrowArgs a,
                                                                           typename Epi::Args ea) {
  __shared__ __attribute__((aligned(16))) uint8_t ring[kRing * kSlot];
  narrow_body<Epi>(a, ea, ring);
}

int narrow_args(NarrowArgs* a, const void* w0_w2, const void* w1, const void* k, const void* v,
                const int32_t* gs, int B, int E, int I, int D, int N, int64_t* blocks,
                const char* what) {
  *a = NarrowArgs{static_cast<const uint16_t*>(w0_w2), static_cast<const uint16_t*>(w1),
                  static_cast<const uint16_t*>(k), static_cast<const uint16_t*>(v), gs, B, E, I, D,
                  N, narrow_m_tiles(I), (N + kTok - 1) / kTok + E, nullptr, 0, 0};
  const int64_t units = ((int64_t)B * a->n_tiles_ub + kXcds - 1) / kXcds * kXcds;
  *blocks = units * a->m_tiles;
  UTTT_REQUIRE(*blocks <= 0x7fffffffLL, "%s: problem too large for one launch", what);
  return UTTT_OK;
}

}  // namespace

// ------------------------------------------------------------------ host ----
bool narrow_experts(int I, int D) { return I <= 512 && D <= 512 && D > kTK; }
bool narrow_stage1(int I, int D, int N, int B, int E) {
  const int64_t weights = (int64_t)6 * B * E * I * D;  // bytes
  return narrow_experts(I, D) ||
         (D > kTK && (int64_t)I * D <= (int64_t)768 * 1536 &&
          (N <= 128 * (int64_t)E || (N <= 256 * (int64_t)E && weights <= (256 << 20))));
}
bool narrow_bwd(int I, int D, int N, int B) {
  return narrow_experts(I, D) && !(I * D >= 448 * 512 && (int64_t)B * N >= 49152);
}
int narrow_m_tiles(int I) { return (I + kHid - 1) / kHid; }

int launch_narrow_stage1(const void* w0_w2, const void* w1, const void* k, const void* v,
                         const void* lr0, const void* lr1, const void* lr2, int lr_dtype,
                         const int32_t* gs, int B, int E, int I, int D, int N, void* dy, void* hid,
                         void* y_save, void* dh_save, hipStream_t st, const char* what) {
  NarrowArgs a;
  int64_t blocks;
  if (int rc = narrow_args(&a, w0_w2, w1, k, v, gs, B, E, I, D, N, &blocks, what)) return rc;
  UTTT_DTYPE_SWITCH_LR(lr_dtype, LR, {
    using S = typename LR::S;
    const typename NarrowS1<LR>::Args ea{
        static_cast<const S*>(lr0),      static_cast<const S*>(lr1),
        static_cast<const S*>(lr2),      static_cast<uint16_t*>(dy),
        static_cast<uint16_t*>(hid),     static_cast<uint16_t*>(y_save),
        static_cast<uint16_t*>(dh_save)};
    hipLaunchKernelGGL((narrow_kernel<NarrowS1<LR>>), dim3((unsigned)blocks), dim3(kTThreads), 0,
                       st, a, ea);
  });
  return check_launch(what);
}

int launch_narrow_gate_up(const void* w0_w2, const void* x, const int32_t* src_rows,
                          long long src_sb, const int32_t* gs, int B, int E, int I, int D, int N,
                          int T, void* hidden, hipStream_t st, const char* what) {
  NarrowArgs a;
  int64_t blocks;
  if (int rc = narrow_args(&a, w0_w2, nullptr, x, nullptr, gs, B, E, I, D, N, &blocks, what))
    return rc;
  a.src = src_rows;
  a.src_sb = src_sb;
  a.T = T;
  hipLaunchKernelGGL((narrow_kernel<NarrowSwiGLU>), dim3((unsigned)blocks), dim3(kTThreads), 0, st,
                     a, NarrowSwiGLU::Args{static_cast<uint16_t*>(hidden)});
  return check_launch(what);
}

int launch_narrow_bwd(const void* gw0_w2, const void* gw1, const void* k, const void* v,
                      const void* lr0, const void* lr1, const void* lr2, int lr_dtype,
                      const int32_t* gs, int B, int E, int I, int D, int N, const void* y_saved,
                      const void* dh_saved, uint16_t* gdh, uint16_t* gx, uint16_t* dx,
                      uint16_t* hlr, float* lr_part, hipStream_t st, const char* what) {
  NarrowArgs a;
  int64_t blocks;
  if (int rc = narrow_args(&a, gw0_w2, gw1, k, v, gs, B, E, I, D, N, &blocks, what)) return rc;
  UTTT_DTYPE_SWITCH_LR(lr_dtype, LR, {
    using S = typename LR::S;
    const typename NarrowBwd<LR>::Args ea{static_cast<const uint16_t*>(y_saved),
                                          static_cast<const uint16_t*>(dh_saved),
                                          static_cast<const S*>(lr0),
                                          static_cast<const S*>(lr1),
                                          static_cast<const S*>(lr2),
                                          gdh,
                                          gx,
                                          dx,
                                          hlr,
                                          lr_part};
    hipLaunchKernelGGL((narrow_kernel<NarrowBwd<LR>>), dim3((unsigned)blocks), dim3(kTThreads), 0,
                       st, a, ea);
  });
  return check_launch(what);
}

}  // namespace uttt
