// Row-wise preprocessing of the fast-weight inputs for gfx950, forward and
// backward: optional silu, then an optional parameter-free norm over each row
// (l2: x / (|x| + 1e-5); rms: x * rsqrt(mean(x^2) + 1e-5)), then an optional
// rotary embedding over blocks of rope_dim features (first half / second
// half pairs, positions from the row's token index plus an offset).
// Reference:
//   _preprocess_update_inputs  uttt_llm/flame/custom_models/uttt_moe/modeling_recurrent_lact.py:630-657
//   q path of the MoE read      ibid. :588-601
//   l2_norm, rms_norm           uttt_llm/flame/custom_models/uttt_moe/ref_base.py:181-195
//   the fast-weight rotary      ref_base.py:342-355 (RotaryEmbedding of rotary.py, bf16 cos / sin
//                               tables of rotary.py:394-433, non-interleaved kernel rotary.py:83-104)
//
// Rounding points are the reference's: F.silu rounds to the storage dtype;
// l2_norm / rms_norm are torch.compile'd, so the norm and the denominator stay
// in fp32 and only the normalised value is rounded to the storage dtype; the
// rotary input is cast to the tables' dtype (bf16), rotated in fp32 with the
// bf16 table values and stored in bf16.  The backward rounds where the
// reference's autograd does: the rotary backward (the conjugate rotation)
// stores bf16, the compiled norm's backward and the silu backward store the
// input dtype.
//
// G lanes (8 to 64, a power of two) per row, NI chunks of 8 elements (one
// 16-byte bf16 vector or two fp32 ones) per lane: chunk i of lane c is c + G i;
// the row stays in registers between the reductions and the element pass, so
// it is read once and written once.  A rotary pair (j, j + R) of a block sits
// R / 8 lanes apart in the same lane step (G is a multiple of a block's 2R / 8
// chunks), so the partner values come from one lane exchange.  Bound by
// memory; with one wave per row and always 8 chunks per lane a 384-element row
// paid the loads and exponentials of 4096: forward with rotary over 16 384 such
// rows 46 us, backward 68, now 15 and 19.
#include <type_traits>

#include "common.h"

namespace uttt {
namespace {

constexpr int kMaxChunksPerLane = 8;  // rows of up to 64 * 8 * 8 = 4096 elements
constexpr int kPrepThreads = 256;

template <class TT>
__device__ __forceinline__ void load8(const typename TT::S* p, float (&v)[8]) {
  if constexpr (sizeof(typename TT::S) == 2) {
    const uint4 u = *reinterpret_cast<const uint4*>(p);
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[2 * k] = TT::load((uint16_t)(w[k] & 0xffffu));
      v[2 * k + 1] = TT::load((uint16_t)(w[k] >> 16));
    }
  } else {
    const float4 a = *reinterpret_cast<const float4*>(p);
    const float4 b = *reinterpret_cast<const float4*>(p + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  }
}

template <class TT>
__device__ __forceinline__ void store8(typename TT::S* p, const float (&v)[8]) {
  if constexpr (sizeof(typename TT::S) == 2) {
    uint4 u;
    u.x = (uint32_t)TT::store(v[0]) | ((uint32_t)TT::store(v[1]) << 16);
    u.y = (uint32_t)TT::store(v[2]) | ((uint32_t)TT::store(v[3]) << 16);
    u.z = (uint32_t)TT::store(v[4]) | ((uint32_t)TT::store(v[5]) << 16);
    u.w = (uint32_t)TT::store(v[6]) | ((uint32_t)TT::store(v[7]) << 16);
    *reinterpret_cast<uint4*>(p) = u;
  } else {
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
    *reinterpret_cast<float4*>(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
  }
}

// the storage dtype's rounding of an fp32 value
template <class TT>
__device__ __forceinline__ float rnd(float x) {
  return TT::load(TT::store(x));
}

template <int G>
__device__ __forceinline__ float row_sum(float v) {
#pragma unroll
  for (int d = G / 2; d > 0; d >>= 1) v += __shfl_xor(v, d, G);
  return v;
}

enum Norm { kNone = 0, kL2 = 1, kRms = 2 };

// Geometry shared by the forward and backward kernels.
struct Rows {
  int64_t rows;
  int D;               // row length (a norm row: a head of q / k, or all of v)
  int64_t ld_in, ld_out;
  int silu, norm;
  // rotary (rope_half = 0: none); table row = token % seq_len + pos_offset
  const uint16_t* cos;  // [table_rows, rope_half] bf16
  const uint16_t* sin;
  int rope_half, rows_per_token, seq_len, pos_offset;
};

// The rotary table row of a row (its token's position); 32-bit divisions where
// the row count fits.
__device__ __forceinline__ int64_t rope_row(const Rows& a, int64_t row) {
  if (a.rows > 0xffffffffLL)  // uniform
    return ((row / a.rows_per_token) % a.seq_len + a.pos_offset) * a.rope_half;
  const uint32_t tok = (uint32_t)row / (uint32_t)a.rows_per_token;
  return (int64_t)((int)(tok % (uint32_t)a.seq_len) + a.pos_offset) * a.rope_half;
}

// The rotary step of one lane step's chunk (8 elements of a row at element
// offset e0 of the row, a multiple of whole blocks into the token): x -> the
// rotated values, with `conj` the conjugate (the backward).  Every lane of the
// group calls it (the exchange is a shuffle); lanes past the row end carry
// values that are never stored.
__device__ __forceinline__ void rope8(float (&x)[8], const Rows& a, int64_t table, int e0,
                                      bool conj) {
  const int R = a.rope_half;     // a power of two
  const int j0 = e0 & (2 * R - 1);
  const bool first = j0 < R;
  const int jj = first ? j0 : j0 - R;
  const uint4 cu = *reinterpret_cast<const uint4*>(a.cos + table + jj);
  const uint4 su = *reinterpret_cast<const uint4*>(a.sin + table + jj);
  const uint32_t cw[4] = {cu.x, cu.y, cu.z, cu.w}, sw[4] = {su.x, su.y, su.z, su.w};
  const int dl = R / 8;  // partner lane distance
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const float c = bf16_to_f32((uint16_t)(u & 1 ? cw[u / 2] >> 16 : cw[u / 2] & 0xffffu));
    float s = bf16_to_f32((uint16_t)(u & 1 ? sw[u / 2] >> 16 : sw[u / 2] & 0xffffu));
    if (conj) s = -s;
    const float p = __shfl_xor(x[u], dl, 64);
    // first half: x0 cos - x1 sin; second half: x0 sin + x1 cos (x0 = partner)
    x[u] = first ? x[u] * c - p * s : p * s + x[u] * c;
  }
}

template <class TI, bool ROPE, int G, int NI>
__global__ __launch_bounds__(kPrepThreads) void rows_prep_kernel(const typename TI::S* __restrict__ in,
                                                        Rows a,
                                                        typename std::conditional<ROPE, BF16T, TI>::type::S* __restrict__ out) {
  using TO = typename std::conditional<ROPE, BF16T, TI>::type;
  const int64_t row0 = (int64_t)blockIdx.x * (kPrepThreads / G) + threadIdx.x / G;
  const bool live = row0 < a.rows;
  const int64_t row = live ? row0 : a.rows - 1;  // every lane takes part in the exchanges
  const int lane = threadIdx.x % G;
  const int chunks = a.D / 8;
  const typename TI::S* src = in + row * a.ld_in;
  typename TO::S* dst = out + row * a.ld_out;
  float v[NI][8];
#pragma unroll
  for (int c = 0; c < NI; ++c) {
    const int ch = lane + G * c;
    // clamped (always valid) address, every load issued before any use
    load8<TI>(src + 8 * (ch < chunks ? ch : chunks - 1), v[c]);
  }
  float ss = 0.0f;
#pragma unroll
  for (int c = 0; c < NI; ++c) {
    const bool ok = lane + G * c < chunks;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      float x = v[c][u];
      if (a.silu) x = rnd<TI>(x / (1.0f + __expf(-x)));
      v[c][u] = x;
      if (ok) ss = __builtin_fmaf(x, x, ss);
    }
  }
  float den = 1.0f, scale = 1.0f;
  if (a.norm == kL2) {
    den = sqrtf(row_sum<G>(ss)) + 1e-5f;
  } else if (a.norm == kRms) {
    scale = __builtin_amdgcn_rsqf(row_sum<G>(ss) / (float)a.D + 1e-5f);
  }
  const int64_t table = ROPE ? rope_row(a, row) : 0;
#pragma unroll
  for (int c = 0; c < NI; ++c) {
    const int ch = lane + G * c;
    float o[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      float y = v[c][u];
      if (a.norm == kL2) y = y / den;
      else if (a.norm == kRms) y = y * scale;
      o[u] = rnd<TI>(y);  // the norm's output, in the input dtype
    }
    if constexpr (ROPE) {
#pragma unroll
      for (int u = 0; u < 8; ++u) o[u] = rnd<BF16T>(o[u]);  // cast to the tables' dtype
      rope8(o, a, table, 8 * (ch < chunks ? ch : chunks - 1), false);
    }
    if (live && ch < chunks) store8<TO>(dst + 8 * ch, o);
  }
}

// grad_in of the row preprocessing given grad_out (the output's dtype):
// conjugate rotation (bf16), the norm's backward on the recomputed silu
// output (fp32, rounded to the input dtype), the silu backward (rounded to
// the input dtype).
template <class TI, bool ROPE, int G, int NI>
__global__ __launch_bounds__(kPrepThreads) void rows_prep_bwd_kernel(
    const typename TI::S* __restrict__ in, Rows a,
    const typename std::conditional<ROPE, BF16T, TI>::type::S* __restrict__ gout,
    typename TI::S* __restrict__ gin) {
  using TO = typename std::conditional<ROPE, BF16T, TI>::type;
  const int64_t row0 = (int64_t)blockIdx.x * (kPrepThreads / G) + threadIdx.x / G;
  const bool live = row0 < a.rows;
  const int64_t row = live ? row0 : a.rows - 1;  // every lane takes part in the exchanges
  const int lane = threadIdx.x % G;
  const int chunks = a.D / 8;
  const typename TI::S* src = in + row * a.ld_in;
  const typename TO::S* gsrc = gout + row * a.ld_out;
  typename TI::S* dst = gin + row * a.ld_in;
  float x[NI][8], g[NI][8];
#pragma unroll
  for (int c = 0; c < NI; ++c) {
    const int ch = lane + G * c;
    const int cc = ch < chunks ? ch : chunks - 1;
    load8<TI>(src + 8 * cc, x[c]);
    load8<TO>(gsrc + 8 * cc, g[c]);
  }
  const int64_t table = ROPE ? rope_row(a, row) : 0;
  float ss = 0.0f, dot = 0.0f;
#pragma unroll
  for (int c = 0; c < NI; ++c) {
    const int ch = lane + G * c;
    const bool ok = ch < chunks;
    if constexpr (ROPE) {
      // the longest rows a chunk at a time (uniform branches; all chunks' rotations
      // interleaved hold too many registers: 16 384 rows of 4096 191 / 249 us)
      if (NI < kMaxChunksPerLane || G * c < chunks) {
        rope8(g[c], a, table, 8 * (ok ? ch : chunks - 1), true);
#pragma unroll
        for (int u = 0; u < 8; ++u) g[c][u] = rnd<TI>(rnd<BF16T>(g[c][u]));
      }
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const float s = a.silu ? rnd<TI>(x[c][u] / (1.0f + __expf(-x[c][u]))) : x[c][u];
      if (ok) {
        ss = __builtin_fmaf(s, s, ss);
        dot = __builtin_fmaf(s, g[c][u], dot);
      }
    }
  }
  float den = 1.0f, coef = 0.0f, scale = 1.0f;
  if (a.norm == kL2) {
    const float n = sqrtf(row_sum<G>(ss));
    dot = row_sum<G>(dot);
    den = n + 1e-5f;
    coef = n > 0.0f ? dot / (n * den * den) : 0.0f;
  } else if (a.norm == kRms) {
    scale = __builtin_amdgcn_rsqf(row_sum<G>(ss) / (float)a.D + 1e-5f);
    dot = row_sum<G>(dot);
    coef = dot * scale * scale * scale / (float)a.D;
  }
#pragma unroll
  for (int c = 0; c < NI; ++c) {
    const int ch = lane + G * c;
    if (!live || ch >= chunks) continue;
    float o[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const float xv = x[c][u];
      const float sg = 1.0f / (1.0f + __expf(-xv));
      const float s = a.silu ? rnd<TI>(xv * sg) : xv;
      float gs = g[c][u];
      if (a.norm == kL2) gs = rnd<TI>(gs / den - s * coef);
      else if (a.norm == kRms) gs = rnd<TI>(scale * gs - s * coef);
      o[u] = a.silu ? gs * (sg * (1.0f + xv * (1.0f - sg))) : gs;
    }
    store8<TI>(dst + 8 * ch, o);
  }
}

int check_rows(const Rows& a, const void* in, const void* out, int dtype, const char* what) {
  UTTT_REQUIRE(a.rows >= 0 && a.D >= 0, "%s: bad sizes rows=%lld D=%d", what, (long long)a.rows,
               a.D);
  UTTT_REQUIRE(in && out, "%s: null pointer", what);
  UTTT_REQUIRE(a.D % 8 == 0 && a.ld_in % 8 == 0 && a.ld_out % 8 == 0 && a.ld_in >= a.D &&
                   a.ld_out >= a.D,
               "%s: D=%d and the row strides must be multiples of 8 (D <= strides)", what, a.D);
  UTTT_REQUIRE(a.D <= 64 * 8 * kMaxChunksPerLane, "%s: D=%d exceeds %d", what, a.D,
               64 * 8 * kMaxChunksPerLane);
  UTTT_REQUIRE(((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 15u) == 0,
               "%s: tensors must be 16-byte aligned", what);
  UTTT_REQUIRE(dtype == UTTT_BF16 || dtype == UTTT_F32 || dtype == UTTT_F16, "%s: dtype code %d",
               what, dtype);
  UTTT_REQUIRE(a.silu == 0 || a.silu == 1, "%s: silu must be 0 or 1", what);
  UTTT_REQUIRE(a.norm == kNone || a.norm == kL2 || a.norm == kRms,
               "%s: norm must be 0 (none), 1 (l2) or 2 (rms)", what);
  UTTT_REQUIRE((a.rows + 3) / 4 <= 0x7fffffffLL, "%s: too many rows", what);
  if (a.rope_half > 0) {
    const int R = a.rope_half;
    UTTT_REQUIRE(R == 8 || R == 16 || R == 32 || R == 64 || R == 128,
                 "%s: rope_dim=%d must be 16, 32, 64, 128 or 256", what, 2 * R);
    UTTT_REQUIRE(a.D % (2 * R) == 0, "%s: rows of D=%d must hold whole rotary blocks of %d", what,
                 a.D, 2 * R);
    UTTT_REQUIRE(a.cos && a.sin && ((reinterpret_cast<uintptr_t>(a.cos) |
                                     reinterpret_cast<uintptr_t>(a.sin)) & 15u) == 0,
                 "%s: rotary tables must be 16-byte aligned", what);
    UTTT_REQUIRE(a.rows_per_token >= 1 && a.seq_len >= 1 && a.pos_offset >= 0,
                 "%s: rows_per_token=%d, seq_len=%d, pos_offset=%d", what, a.rows_per_token,
                 a.seq_len, a.pos_offset);
    UTTT_REQUIRE(a.rows % ((int64_t)a.rows_per_token * a.seq_len) == 0,
                 "%s: %lld rows are not whole sequences of %d tokens x %d rows", what,
                 (long long)a.rows, a.seq_len, a.rows_per_token);
  }
  return UTTT_OK;
}

Rows make_rows(int64_t rows, int D, int64_t ld_in, int64_t ld_out, int silu, int norm,
               const void* cos, const void* sin, int rope_dim, int rows_per_token, int seq_len,
               int pos_offset) {
  Rows a;
  a.rows = rows;
  a.D = D;
  a.ld_in = ld_in;
  a.ld_out = ld_out;
  a.silu = silu;
  a.norm = norm;
  a.cos = static_cast<const uint16_t*>(cos);
  a.sin = static_cast<const uint16_t*>(sin);
  a.rope_half = rope_dim > 0 ? rope_dim / 2 : 0;
  a.rows_per_token = rows_per_token;
  a.seq_len = seq_len;
  a.pos_offset = pos_offset;
  return a;
}

// f(G, NI): the fewest lanes per row (at least 8 and whole rotary blocks) that
// hold it in at most four chunks each, rounded up to a compiled chunk count; of
// few rows more lanes, a chunk each (up to 1000 rows of 512, backward with rotary,
// four chunks on 16 lanes 9.1 us, one on 64 4.3).
template <class F>
void prep_dispatch(int64_t rows, int D, int rope_half, F&& f) {
  const int CH = D / 8, block = rope_half / 4;
  int g = 8;
  while (g < 64 && (4 * g < CH || g < block || (g < CH && rows * g <= 32768))) g *= 2;
  const int ni = (CH + g - 1) / g;
  auto with = [&](auto G) {
    if (ni <= 1) f(G, std::integral_constant<int, 1>{});
    else if (ni <= 3) f(G, std::integral_constant<int, 3>{});
    else f(G, std::integral_constant<int, 4>{});
  };
  switch (g) {
    case 8: with(std::integral_constant<int, 8>{}); break;
    case 16: with(std::integral_constant<int, 16>{}); break;
    case 32: with(std::integral_constant<int, 32>{}); break;
    default:
      if (ni > 4)
        f(std::integral_constant<int, 64>{}, std::integral_constant<int, kMaxChunksPerLane>{});
      else
        with(std::integral_constant<int, 64>{});
  }
}
inline unsigned prep_blocks(int64_t rows, int g) {
  const int per = kPrepThreads / g;
  return (unsigned)((rows + per - 1) / per);
}

}  // namespace
}  // namespace uttt

using namespace uttt;

extern "C" int uttt_rows_preprocess(const void* in, int dtype, int64_t rows, int D, int64_t ld_in,
                                    int silu, int norm, const void* rope_cos,
                                    const void* rope_sin, int rope_dim, int rows_per_token,
                                    int seq_len, int pos_offset, int table_rows, void* out,
                                    int64_t ld_out, void* stream) {
  const Rows a = make_rows(rows, D, ld_in, ld_out, silu, norm, rope_cos, rope_sin, rope_dim,
                           rows_per_token, seq_len, pos_offset);
  if (rows == 0 || D == 0) return UTTT_OK;
  if (int rc = check_rows(a, in, out, dtype, "rows_preprocess")) return rc;
  UTTT_REQUIRE(rope_dim == 0 || pos_offset + seq_len <= table_rows,
               "rows_preprocess: positions up to %d past the rotary table's %d rows",
               pos_offset + seq_len, table_rows);
  hipStream_t st = as_stream(stream);
  UTTT_DTYPE_SWITCH_LR(dtype, TT, {
    using S = typename TT::S;
    prep_dispatch(rows, D, a.rope_half, [&](auto g, auto ni) {
      constexpr int G = decltype(g)::value, NI = decltype(ni)::value;
      const dim3 grid(prep_blocks(rows, G));
      if (rope_dim > 0)
        hipLaunchKernelGGL((rows_prep_kernel<TT, true, G, NI>), grid, dim3(kPrepThreads), 0, st,
                           static_cast<const S*>(in), a, static_cast<uint16_t*>(out));
      else
        hipLaunchKernelGGL((rows_prep_kernel<TT, false, G, NI>), grid, dim3(kPrepThreads), 0, st,
                           static_cast<const S*>(in), a, static_cast<S*>(out));
    });
  });
  return check_launch("rows_preprocess");
}

extern "C" int uttt_rows_preprocess_bwd(const void* in, int dtype, const void* grad_out,
                                        int64_t rows, int D, int64_t ld_in, int64_t ld_out,
                                        int silu, int norm, const void* rope_cos,
                                        const void* rope_sin, int rope_dim, int rows_per_token,
                                        int seq_len, int pos_offset, int table_rows,
                                        void* grad_in, void* stream) {
  const Rows a = make_rows(rows, D, ld_in, ld_out, silu, norm, rope_cos, rope_sin, rope_dim,
                           rows_per_token, seq_len, pos_offset);
  if (rows == 0 || D == 0) return UTTT_OK;
  if (int rc = check_rows(a, in, grad_in, dtype, "rows_preprocess_bwd")) return rc;
  UTTT_REQUIRE(grad_out && (reinterpret_cast<uintptr_t>(grad_out) & 15u) == 0,
               "rows_preprocess_bwd: grad_out must be a 16-byte aligned tensor");
  UTTT_REQUIRE(rope_dim == 0 || pos_offset + seq_len <= table_rows,
               "rows_preprocess_bwd: positions up to %d past the rotary table's %d rows",
               pos_offset + seq_len, table_rows);
  hipStream_t st = as_stream(stream);
  UTTT_DTYPE_SWITCH_LR(dtype, TT, {
    using S = typename TT::S;
    prep_dispatch(rows, D, a.rope_half, [&](auto g, auto ni) {
      constexpr int G = decltype(g)::value, NI = decltype(ni)::value;
      const dim3 grid(prep_blocks(rows, G));
      if (rope_dim > 0)
        hipLaunchKernelGGL((rows_prep_bwd_kernel<TT, true, G, NI>), grid, dim3(kPrepThreads), 0, st,
                           static_cast<const S*>(in), a, static_cast<const uint16_t*>(grad_out),
                           static_cast<S*>(grad_in));
      else
        hipLaunchKernelGGL((rows_prep_bwd_kernel<TT, false, G, NI>), grid, dim3(kPrepThreads), 0,
                           st, static_cast<const S*>(in), a, static_cast<const S*>(grad_out),
                           static_cast<S*>(grad_in));
    });
  });
  return check_launch("rows_preprocess_bwd");
}
