// bf16 MFMA products on 192 x 192 tiles, two workgroups per CU (gfx950).
//
// The 256 x 256 pipeline of gemm_pipe.h owns a whole CU (128 KiB of LDS, 256
// accumulators per lane) and pays one prologue and one epilogue per tile with
// the matrix cores idle.  That is right for long reductions of wide matrices;
// with sides of 192 or 384 (the shipped expert and head widths) a tile
// multiplies 6 to 12 short steps, half of them padding.  Here a workgroup of
// four waves (2 x 2, 96 x 96 outputs each: 3 x 3 blocks of
// v_mfma_f32_32x32x16_bf16, 144 accumulators per lane) streams stages of 32 k
// through a three-slot LDS ring of 24 KiB slots: 72 KiB, so two workgroups
// share a CU and one's loads, waits and epilogue run under the other's
// products.  Every width of the model family (192, 384, 768, 1536, 3072) is a
// whole number of tiles.  A wave reads 6 fragments per 9 MFMAs.
//
// LDS layouts (16-byte chunks, filled by buffer_load ... lds, 1 KiB per wave
// instruction):
//   KMajor (rows of 32 k = 64 bytes, 4 chunks): chunk c of row r in slot
//     4 r + (c ^ ((r >> 2) & 3)).  16 consecutive rows of one chunk cover all
//     64 banks once.
//   RMajor (32 k-rows of 192 elements = 384 bytes, 24 chunks): the 64-byte
//     block b (4 chunks) of k-row k in block b ^ ((k >> 1) & 1).  A transposing
//     read touches one block of 4 consecutive k-rows; 384 = 256 + 128, so
//     k-rows k and k + 2 would share banks without the exchange.
#pragma once

#include <type_traits>

#include "gemm_pipe.h"

namespace uttt {
namespace t192 {

using namespace pipe;

constexpr int kT = 192;                  // tile rows of either operand
constexpr int kTK = 32;                  // k per stage
constexpr int kWT = kT / 2;              // outputs per wave along each side
constexpr int kNBlk = kWT / 32;          // 3 x 3 MFMA blocks per wave
constexpr int kTTile = kT * kTK * 2;     // 12 KiB
constexpr int kTStage = 2 * kTTile;
constexpr int kTRing = 3;
constexpr int kTThreads = 256;
constexpr int kTLoads = kTTile / 16 / kTThreads;  // 3 loads per wave and operand tile
constexpr int kTItems = kWT * (kT / 8) / kTThreads;  // epilogue items per thread and half

// The loads of one operand's tile of ROWS rows over a K loop (see TileLoader in
// gemm_pipe.h: rows past the end repeat the last valid row, k past the end
// reads zeros through the descriptor's record bound).  `split` (KMajor): tile
// rows from `split` on are the operand's rows r0 .. again, `second` elements
// further on (two row blocks of one matrix in one tile).
template <int MAJOR, int ROWS = kT>
struct Loader {
  static constexpr int kLoads = ROWS * kTK * 2 / 16 / kTThreads;
  const uint8_t* base;
  int64_t kstep;
  int last, k_end, ld2, col2;
  uint32_t off[kLoads];
  int wofs;

  __device__ __forceinline__ void init(const Operand& op, int r0, int split = ROWS,
                                       int second = 0) {
    const int lane = threadIdx.x & 63;
    const int w = wave_id();
    k_end = op.k_end;
    last = (op.k_end + kTK - 1) / kTK - 1;
    wofs = w * 1024;
    asm volatile("" : "+s"(wofs));
    ld2 = (int)op.ld * 2;
    int nrows = op.r_end - r0;
    const uint16_t* org;
    if (nrows > 0) {
      org = MAJOR == KMajor ? op.base + (int64_t)r0 * op.ld : op.base + r0;
      col2 = r0 * 2;
    } else {  // no valid row: read the operand's first rows instead
      org = op.base;
      nrows = MAJOR == KMajor ? 1 : 8;
      col2 = 0;
    }
    base = uniform_ptr(reinterpret_cast<const uint8_t*>(org));
    kstep = MAJOR == KMajor ? (int64_t)kTK * 2 : (int64_t)kTK * op.ld * 2;
#pragma unroll
    for (int t = 0; t < kLoads; ++t) {
      const int s = (t * 4 + w) * 64 + lane;
      if constexpr (MAJOR == KMajor) {
        const int r = s >> 2;
        const int c = (s & 3) ^ ((r >> 2) & 3);
        const int rr = r < split ? r : r - split;
        off[t] = (uint32_t)((rr < nrows ? rr : nrows - 1) * (int)op.ld + c * 8 +
                            (r < split ? 0 : second)) * 2u;
      } else {
        const int k = s / (ROWS / 8), cc = s - k * (ROWS / 8);
        const int c = cc ^ (((k >> 1) & 1) << 2);
        const int cmax = (nrows >> 3) - 1;
        off[t] = (uint32_t)(k * (int)op.ld + (c < cmax ? c : cmax) * 8) * 2u;
      }
      asm volatile("" : "+v"(off[t]));
    }
  }

  // A KMajor tile of gathered rows: row(r) of org for tile row r (below 2^30
  // elements in).
  template <class Row>
  __device__ __forceinline__ void init_gather(const uint16_t* org, int ld, int k_end_, Row&& row) {
    const int lane = threadIdx.x & 63;
    const int w = wave_id();
    k_end = k_end_;
    last = (k_end + kTK - 1) / kTK - 1;
    wofs = w * 1024;
    asm volatile("" : "+s"(wofs));
    base = uniform_ptr(reinterpret_cast<const uint8_t*>(org));
    kstep = (int64_t)kTK * 2;
#pragma unroll
    for (int t = 0; t < kLoads; ++t) {
      const int s = (t * 4 + w) * 64 + lane;
      const int r = s >> 2;
      off[t] = (uint32_t)(row(r) * ld + ((s & 3) ^ ((r >> 2) & 3)) * 8) * 2u;
      asm volatile("" : "+v"(off[t]));
    }
  }

  // Step `step` (0 .. last, in order) into the tile at LDS `dst`.
  __device__ __forceinline__ void issue(int step, uint8_t* dst) {
    const uint8_t* sb = uniform_ptr(base + (int64_t)step * kstep);
    uint32_t recs = 0xFFFFFFFFu;
    if (step == last && (k_end % kTK) != 0) {
      if constexpr (MAJOR == RMajor) {
        recs = (uint32_t)((k_end - step * kTK) * ld2 - col2);
      } else {
        // lanes past k_end go past the bound; valid offsets (192 rows of under
        // 2^23 elements) stay below it
        recs = 0xFFFFFF00u;
        const int lane = threadIdx.x & 63, w = wofs >> 10, kt = k_end % kTK;
#pragma unroll
        for (int t = 0; t < kLoads; ++t) {
          const int sl = (t * 4 + w) * 64 + lane;
          const int r = sl >> 2;
          if (((sl & 3) ^ ((r >> 2) & 3)) * 8 >= kt) off[t] = 0xFFFFFFF0u;
        }
      }
    }
    const Rsrc rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(sb), (short)0,
                                                      (int)recs, kBufferWord3);
#pragma unroll
    for (int t = 0; t < kLoads; ++t)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, UTTT_LDS(dst + t * 4096 + wofs), 16, off[t], 0,
                                               0, 0);
  }
};

// This lane's LDS byte offsets of a wave's three 32-row fragments in a tile.
// KMajor: one offset per k-substep, the row blocks 2048 bytes apart.
// RMajor: one offset per row block, the substep 6144 bytes on and the second
// transposing read 1536 (4 k-rows).
template <int MAJOR>
struct FragAddr {
  uint32_t a[MAJOR == KMajor ? 2 : kNBlk];
  __device__ __forceinline__ void init(int wrow) {  // wrow: 0 or 1, the wave's half of the rows
    const int lane = threadIdx.x & 63;
    if constexpr (MAJOR == KMajor) {
      const int r = lane & 31;
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
        a[ks] = (uint32_t)(wrow * kWT * 64 +
                           (r * 4 + ((2 * ks + (lane >> 5)) ^ ((r >> 2) & 3))) * 16);
    } else {
      const int g = lane >> 4, s = lane & 15, j = s >> 2, q = s & 3;
      const int k0 = 8 * (g >> 1) + j, x = (j >> 1) & 1;
#pragma unroll
      for (int i = 0; i < kNBlk; ++i)
        a[i] = (uint32_t)(k0 * 384 + (4 * ((kNBlk * wrow + i) ^ x) + 2 * (g & 1) + (q >> 1)) * 16 +
                          8 * (q & 1));
    }
  }
  template <int KS, int I>
  __device__ __forceinline__ bf16x8 read(uint32_t tile) const {
    if constexpr (MAJOR == KMajor) {
      return ds_b128_asm<I * 2048>(tile + a[KS]);
    } else {
      const i16x4 x0 = ds_tr16_asm<KS * 6144>(tile + a[I]);
      const i16x4 x1 = ds_tr16_asm<KS * 6144 + 1536>(tile + a[I]);
      return __builtin_bit_cast(bf16x8, __builtin_shufflevector(x0, x1, 0, 1, 2, 3, 4, 5, 6, 7));
    }
  }
};

struct Frags {
  bf16x8 a[kNBlk], b[kNBlk];
};

// s_waitcnt lgkmcnt(N) that redefines the fragment registers (no MFMA that
// reads them can move above it).
template <int N>
__device__ __forceinline__ void wait_frags(Frags& f) {
  i32x4 r[6];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    r[i] = __builtin_bit_cast(i32x4, f.a[i]);
    r[3 + i] = __builtin_bit_cast(i32x4, f.b[i]);
  }
  asm volatile("s_waitcnt lgkmcnt(%6)"
               : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]), "+v"(r[4]), "+v"(r[5])
               : "i"(N)
               : "memory");
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    f.a[i] = __builtin_bit_cast(bf16x8, r[i]);
    f.b[i] = __builtin_bit_cast(bf16x8, r[3 + i]);
  }
}

// bf16(c * x) of a fragment.
__device__ __forceinline__ bf16x8 scaled(const bf16x8& x, float c) {
  i32x4 w = __builtin_bit_cast(i32x4, x);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t u = (uint32_t)w[k];
    w[k] = (int)pack_bf16x2(c * __uint_as_float(u << 16), c * __uint_as_float(u & 0xffff0000u));
  }
  return __builtin_bit_cast(bf16x8, w);
}

typedef f32x16 Acc[kNBlk][kNBlk];

__device__ __forceinline__ void mma9(Acc& acc, const Frags& f) {
  static_for<kNBlk * kNBlk>([&](auto Q) __attribute__((always_inline)) {
    constexpr int i = decltype(Q)::value / kNBlk, j = decltype(Q)::value % kNBlk;
    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a[i], f.b[j], acc[i][j], 0, 0, 0);
  });
}

// acc += A B^T over nk >= 1 stages.  Stage k: wait for its loads (stage k+1's
// stay in flight), barrier (stage k landed for every wave; every wave is done
// with the slot of stage k-1), issue stage k+2 into that slot, read both
// k-substeps' fragments, multiply.  All LDS reads are inline asm with explicit
// waits (the compiler would drain the loads in flight in front of them).  The
// products run in increasing k in 16-wide steps with A in the first operand,
// as in gemm_pipe.h, so the results are the 256-tile kernels' bits.
// SCALE_B: the second operand is bf16(b_scale * B), converted as its
// fragments are read.  at(k), run before stage k is issued, gives the loaders'
// step of it (a chained second pair points them at its operands there).
struct SameStep {
  __device__ int operator()(int k) const { return k; }
};
template <int AMAJ, int BMAJ, bool SCALE_B = false, class At = SameStep>
__device__ __forceinline__ void k_loop(Loader<AMAJ>& la, Loader<BMAJ>& lb, int nk, uint8_t* ring,
                                       Acc& acc, float b_scale = 1.0f, At&& at = At()) {
  const int w = wave_id();
  FragAddr<AMAJ> fa;
  FragAddr<BMAJ> fb;
  fa.init(w >> 1);
  fb.init(w & 1);
  constexpr int kOps = kNBlk * (AMAJ == KMajor ? 1 : 2) + kNBlk * (BMAJ == KMajor ? 1 : 2);
  uint8_t *p0 = ring, *p1 = ring + kTStage, *p2 = ring + 2 * kTStage;
  auto issue = [&](int k, uint8_t* slot) __attribute__((always_inline)) {
    const int step = at(k);
    la.issue(step, slot);
    lb.issue(step, slot + kTTile);
  };
  issue(0, p0);
  if (nk > 1) issue(1, p1);
  Frags f[2];
  for (int k = 0; k < nk; ++k) {
    if (k + 1 < nk)
      wait_vmcnt<2 * kTLoads>();
    else
      wait_vmcnt<0>();
    block_barrier();
    __builtin_amdgcn_sched_barrier(0);
    const uint32_t ta = lds_addr(p0), tb = ta + kTTile;
    static_for<2>([&](auto KS) __attribute__((always_inline)) {
      static_for<kNBlk>([&](auto I) __attribute__((always_inline)) {
        f[KS].a[I] = fa.template read<decltype(KS)::value, decltype(I)::value>(ta);
        f[KS].b[I] = fb.template read<decltype(KS)::value, decltype(I)::value>(tb);
      });
    });
    if (k + 2 < nk) issue(k + 2, p2);
    __builtin_amdgcn_sched_barrier(0);
    wait_frags<kOps>(f[0]);
    if constexpr (SCALE_B)
      static_for<kNBlk>([&](auto I) __attribute__((always_inline)) { f[0].b[I] = scaled(f[0].b[I], b_scale); });
    mma9(acc, f[0]);
    __builtin_amdgcn_sched_barrier(0);
    wait_frags<0>(f[1]);
    if constexpr (SCALE_B)
      static_for<kNBlk>([&](auto I) __attribute__((always_inline)) { f[1].b[I] = scaled(f[1].b[I], b_scale); });
    mma9(acc, f[1]);
    __builtin_amdgcn_sched_barrier(0);
    uint8_t* t = p0;
    p0 = p1;
    p1 = p2;
    p2 = t;
  }
}

__device__ __forceinline__ void zero_acc(Acc& acc) {
  static_for<kNBlk * kNBlk>([&](auto Q) __attribute__((always_inline)) {
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[Q / kNBlk][Q % kNBlk][v] = 0.0f;
  });
}

// Epilogue frame: one 96-column half of the tile at a time, the two waves that
// own it write it to LDS as fp32 [column][192 rows] (the ring, free after the K
// loop; 16-byte chunks XOR-swizzled by column), then thread t takes column
// it / 24 and rows 8 (it % 24) .. + 7 for it = t, t + 256, ...: 24 lanes cover
// the 192 rows of a column, 384 contiguous bytes of bf16 output.
//   before(h, k, n, g) runs for each item before its half is staged (loads),
//   body(h, k, n, g, v[8]) after; k = 0 .. kTItems - 1, n = column in the tile.
// With `transposed` (wave-uniform) the half is then read along the other side:
// body's results (v as it leaves them) go back to LDS, and across(r, n, v[8])
// gets columns n .. n + 7 of tile row r (consecutive lanes on consecutive rows:
// conflict-free reads; the 16-byte stores of a row meet in L2).
struct NoAcross {
  __device__ void operator()(int, int, const float (&)[8]) const {}
};
template <class Before, class Body, class Across = NoAcross>
__device__ __forceinline__ void staged(const Acc& acc, float* lds, Before&& before, Body&& body,
                                       bool transposed = false, Across&& across = Across()) {
  const int w = wave_id();
  const int wm = w >> 1, wn = w & 1;
  block_barrier();  // every wave is done reading the ring
  static_for<2>([&](auto H) __attribute__((always_inline)) {
    constexpr int h = H;
    static_for<kTItems>([&](auto K) __attribute__((always_inline)) {
      const int it = threadIdx.x + kTThreads * K;
      before(H, K, h * kWT + it / 24, it % 24);
    });
    if (wn == h) {
      static_for<kNBlk * kNBlk * 4>([&](auto Q) __attribute__((always_inline)) {
        constexpr int i = decltype(Q)::value / (kNBlk * 4), j = (decltype(Q)::value / 4) % kNBlk,
                      q = decltype(Q)::value % 4;
        const int n = j * 32 + acc_col();
        const int c = (wm * kWT + i * 32 + acc_row(q * 4)) >> 2;
        *reinterpret_cast<float4*>(lds + n * kT + ((c ^ (n & 15)) << 2)) =
            make_float4(acc[i][j][q * 4], acc[i][j][q * 4 + 1], acc[i][j][q * 4 + 2],
                        acc[i][j][q * 4 + 3]);
      });
    }
    block_barrier();
    static_for<kTItems>([&](auto K) __attribute__((always_inline)) {
      const int it = threadIdx.x + kTThreads * K;
      const int n = it / 24, g = it % 24;
      float4* pa = reinterpret_cast<float4*>(lds + n * kT + (((2 * g) ^ (n & 15)) << 2));
      float4* pb = reinterpret_cast<float4*>(lds + n * kT + (((2 * g + 1) ^ (n & 15)) << 2));
      const float4 a = *pa, b = *pb;
      float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
      body(H, K, h * kWT + n, g, v);
      if constexpr (!std::is_same_v<std::decay_t<Across>, NoAcross>) {
        if (transposed) {
          *pa = make_float4(v[0], v[1], v[2], v[3]);
          *pb = make_float4(v[4], v[5], v[6], v[7]);
        }
      }
    });
    if constexpr (!std::is_same_v<std::decay_t<Across>, NoAcross>) {
      if (transposed) {
        block_barrier();
#pragma unroll 1
        for (int k = 0; k < kTItems; ++k) {
          const int it = threadIdx.x + kTThreads * k;
          const int r = it % kT, n = it / kT * 8;
          float v[8];
#pragma unroll
          for (int u = 0; u < 8; ++u)
            v[u] = lds[(n + u) * kT + (((r >> 2) ^ ((n + u) & 15)) << 2) + (r & 3)];
          across(r, h * kWT + n, v);
        }
      }
    }
    if (h == 0) block_barrier();
  });
}

}  // namespace t192
}  // namespace uttt
