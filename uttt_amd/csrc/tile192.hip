// Products of narrow matrices on 192 x 192 tiles (tile192.h): the weight
// gradients of small experts, their token segments cut into chunks, and the
// Newton-Schulz steps of mid-sized matrices.  Called through the C entries of
// grouped_gemm.hip, which choose between these and the 256 x 256 tiles.
#include <algorithm>

#include "tile192.h"
#include "tile192_host.h"

namespace uttt {
namespace {

using namespace pipe;
using namespace t192;

__device__ __forceinline__ void store8_bf16(uint16_t* p, const float (&v)[8]) {
  uint4 u;
  u.x = pack_bf16x2(v[0], v[1]);
  u.y = pack_bf16x2(v[2], v[3]);
  u.z = pack_bf16x2(v[4], v[5]);
  u.w = pack_bf16x2(v[6], v[7]);
  *reinterpret_cast<uint4*>(p) = u;
}

__device__ __forceinline__ void unpack8_bf16(const uint4& u, float (&v)[8]) {
  const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    v[2 * k] = bf16_to_f32((uint16_t)(w[k] & 0xffffu));
    v[2 * k + 1] = bf16_to_f32((uint16_t)(w[k] >> 16));
  }
}

// This workgroup's place among n when every XCD takes a contiguous eighth of
// them (grid xcd_run_blocks(n)), or -1: neighbours share an XCD's L2, and few
// large groups still reach every XCD.
__device__ __forceinline__ int xcd_run(int n) {
  const int each = (n + kXcds - 1) / kXcds;
  const int i = blockIdx.x % kXcds * each + blockIdx.x / kXcds;
  return i < n ? i : -1;
}
int64_t xcd_run_blocks(int64_t n) { return (n + kXcds - 1) / kXcds * kXcds; }

// ======================================================= weight gradients ==
// out[b, e][x][y] = sum_{n in seg(b, e)} P[n, y] Q[n, x] (two tasks per
// launch), the segment of every expert cut into chunks of `chunk` tokens: one
// workgroup per (chunk, output tile).  An expert with one chunk (an empty one
// has one of no tokens: zeros) stores its bf16 output; the chunks of a longer
// one store fp32 partials, part[b * parts_ub + index among the batch's partial
// chunks], which wg192_reduce_kernel adds in chunk order (the result does not
// depend on scheduling).  An expert with several chunks has more than `chunk`
// tokens, so a batch has at most 2 N / chunk partial chunks.
//
// Bound by the token rows' stream from memory: 48 experts of 192 x 192 over
// 196 608 tokens read 377 MB in 98 us (+ 6 us of reduction), against 285-459 us
// (routing from even to skewed) for one 256 x 256-tile workgroup per output
// tile, where 144 workgroups run and the longest expert sets the time; 96
// experts of 384 x 384 over 16 384 tokens 42 us against 70.
struct Wg192Task {
  const uint16_t* p;
  const uint16_t* q;
  uint16_t* out;
  int X, Y;
  int y_tiles, x_tiles;
};

struct Wg192Args {
  Wg192Task t[2];
  const int32_t* gs;
  float* part;       // [B * parts_ub][n_out] fp32
  int64_t n_out;     // elements of both outputs of one expert
  int B, E, N, chunk;
  int slots, parts_ub;  // upper bounds of one batch's chunks and partial chunks
  int run;              // tiles of one chunk that run on one XCD
};

// Chunk `slot` of a batch: its expert, first token, tokens, and its index
// among the partial chunks (-1: the expert's only chunk).
struct ChunkPos {
  int e, start, size, part;
};

// The chunks of a segment of g tokens, and those that store partials.
__device__ __forceinline__ int chunks_of(int g, int chunk) { return max(1, (g + chunk - 1) / chunk); }
__device__ __forceinline__ int partials_of(int nt) { return nt > 1 ? nt : 0; }

__device__ ChunkPos find_chunk(const int32_t* __restrict__ gs_b, int E, int N, int chunk,
                               int slot) {
  const int lane = threadIdx.x & 63;
  int tok_base = 0, base = 0, pbase = 0;
  for (int e0 = 0; e0 < E; e0 += 64) {
    const int e = e0 + lane;
    const int graw = e < E ? gs_b[e] : 0;
    const int g = graw > 0 ? graw : 0;
    const int tok_incl = wave_incl_scan(g);
    const int start = min(tok_base + tok_incl - g, N);
    const int gc = min(g, N - start);
    const int nt = e < E ? chunks_of(gc, chunk) : 0;
    const int incl = wave_incl_scan(nt);
    const int excl = base + incl - nt;
    const int pincl = wave_incl_scan(partials_of(nt));
    const uint64_t bal = __ballot(slot >= excl && slot < excl + nt);
    if (bal != 0ull) {
      const int src = __ffsll((unsigned long long)bal) - 1;
      const int i = slot - lane_value(excl, src);
      const int size = lane_value(gc, src) - i * chunk;
      const int parts = lane_value(nt, src);
      return ChunkPos{__builtin_amdgcn_readfirstlane(e0 + src), lane_value(start, src) + i * chunk,
                      min(size, chunk),
                      parts > 1 ? pbase + lane_value(pincl, src) - parts + i : -1};
    }
    tok_base += lane_value(tok_incl, 63);
    base += lane_value(incl, 63);
    pbase += lane_value(pincl, 63);
  }
  return ChunkPos{-1, 0, 0, -1};
}

__global__ __launch_bounds__(kTThreads, 2) void wg192_kernel(Wg192Args a) {
  __shared__ __attribute__((aligned(16))) uint8_t ring[kTRing * kTStage];
  const int n0 = a.t[0].y_tiles * a.t[0].x_tiles;
  const int per = n0 + a.t[1].y_tiles * a.t[1].x_tiles;
  // the tiles of one chunk run on one XCD (they read the same token rows), or,
  // of few chunks, in runs of a.run tiles dealt to the XCDs
  const int loc = blockIdx.x / kXcds, runs = (per + a.run - 1) / a.run;
  const int r = loc / a.run * kXcds + blockIdx.x % kXcds;
  const int unit = r / runs, t = r % runs * a.run + loc % a.run;
  if (unit >= a.B * a.slots || t >= per) return;
  const int b = unit / a.slots;
  const ChunkPos cp = find_chunk(a.gs + (int64_t)b * a.E, a.E, a.N, a.chunk, unit - b * a.slots);
  if (cp.e < 0) return;
  const bool first = t < n0;
  const Wg192Task& tk = first ? a.t[0] : a.t[1];
  const int tl = first ? t : t - n0;
  const int y0 = tl / tk.x_tiles * kT, x0 = tl % tk.x_tiles * kT;
  Acc acc;
  zero_acc(acc);
  if (cp.size > 0) {
    const int64_t row = (int64_t)b * a.N + cp.start;
    const Operand P{tk.p + row * tk.Y, tk.Y, tk.Y, cp.size};
    const Operand Q{tk.q + row * tk.X, tk.X, tk.X, cp.size};
    Loader<RMajor> lp, lq;
    lp.init(P, y0);
    lq.init(Q, x0);
    k_loop<RMajor, RMajor>(lp, lq, (cp.size + kTK - 1) / kTK, ring, acc);
  }
  const int X = tk.X, Y = tk.Y;
  const bool partial = cp.part >= 0;
  uint16_t* out = tk.out + ((int64_t)b * a.E + cp.e) * X * Y;
  float* part = a.part + ((int64_t)b * a.parts_ub + (partial ? cp.part : 0)) * a.n_out + (first ? 0 : (int64_t)a.t[0].X * a.t[0].Y);
  staged(
      acc, reinterpret_cast<float*>(ring), [](auto, auto, int, int) {},
      [&](auto, auto, int n, int g, float (&v)[8]) __attribute__((always_inline)) {
        const int x = x0 + n, y = y0 + 8 * g;
        if (x >= X || y >= Y) return;
        const int64_t at = (int64_t)x * Y + y;
        if (partial) {
          *reinterpret_cast<float4*>(part + at) = make_float4(v[0], v[1], v[2], v[3]);
          *reinterpret_cast<float4*>(part + at + 4) = make_float4(v[4], v[5], v[6], v[7]);
        } else {
          store8_bf16(out + at, v);
        }
      });
}

// The outputs of the experts with several chunks: bf16 of the partials' sum,
// added in chunk order.  `each` workgroups per (b, e), in one grid axis (the
// others end at 65 535, which B * E need not).
__global__ __launch_bounds__(256) void wg192_reduce_kernel(Wg192Args a, int each) {
  const int be = blockIdx.x / each, blk = blockIdx.x % each;
  const int b = be / a.E, e = be % a.E;
  const int lane = threadIdx.x & 63;
  const int32_t* gs_b = a.gs + (int64_t)b * a.E;
  int tok_base = 0, slot = 0, parts = 0;
  for (int e0 = 0; e0 < a.E; e0 += 64) {
    const int ee = e0 + lane;
    const int graw = ee < a.E ? gs_b[ee] : 0;
    const int g = graw > 0 ? graw : 0;
    const int tok_incl = wave_incl_scan(g);
    const int start = min(tok_base + tok_incl - g, a.N);
    const int nt = ee < a.E ? partials_of(chunks_of(min(g, a.N - start), a.chunk)) : 0;
    const int incl = wave_incl_scan(nt);
    if (e < e0 + 64) {
      parts = lane_value(nt, e - e0);
      slot += lane_value(incl, e - e0) - parts;
      break;
    }
    tok_base += lane_value(tok_incl, 63);
    slot += lane_value(incl, 63);
  }
  if (parts < 2) return;
  const int64_t n0 = (int64_t)a.t[0].X * a.t[0].Y;
  const float* src = a.part + ((int64_t)b * a.parts_ub + slot) * a.n_out;
  for (int64_t i = ((int64_t)blk * 256 + threadIdx.x) * 8; i < a.n_out; i += (int64_t)each * 2048) {
    float v[8] = {};
#pragma unroll 4
    for (int s = 0; s < parts; ++s) {
      const float4 x = *reinterpret_cast<const float4*>(src + s * a.n_out + i);
      const float4 y = *reinterpret_cast<const float4*>(src + s * a.n_out + i + 4);
      v[0] += x.x; v[1] += x.y; v[2] += x.z; v[3] += x.w;
      v[4] += y.x; v[5] += y.y; v[6] += y.z; v[7] += y.w;
    }
    uint16_t* o = i < n0 ? a.t[0].out + ((int64_t)b * a.E + e) * n0 + i
                         : a.t[1].out + ((int64_t)b * a.E + e) * (a.n_out - n0) + i - n0;
    store8_bf16(o, v);
  }
}

// ================================================= token-grouped products ==
// y[b, n, m] = sum_k A(m, k) x[b, n, k] (+ a second pair chained along k) over
// the tokens n of each expert, A [M, K] (KMajor) or [K, M] (RMajor) per expert;
// bf16, the 256-token kernels' bits.  For narrow experts the token rows' stream
// bounds it: 48 of 192 x 192 over 196 608 tokens 377 MB in 88 us (grad_K), 226
// in 55 (grad_V).  Super-tiles as in tn_kernel, 64 workgroups to an XCD at once.
struct Tn192Args {
  const uint16_t* a[2];
  const uint16_t* x[2];
  int K[2];  // K[1] = 0: one product
  uint16_t* y;
  const int32_t* gs;
  int B, E, N, M, m_tiles, n_tiles_ub;
  int gm, gn, n_super_m;  // super-tiles: gm m-tiles x gn token tiles on one XCD
};

template <int AMAJ>
__global__ __launch_bounds__(kTThreads, 2) void tn192_kernel(Tn192Args s) {
  __shared__ __attribute__((aligned(16))) uint8_t ring[kTRing * kTStage];
  const int loc = blockIdx.x / kXcds, per = s.gm * s.gn;
  const int sup = loc / per * kXcds + blockIdx.x % kXcds, p = loc % per;
  const int mt = sup % s.n_super_m * s.gm + p % s.gm;
  const int unit = sup / s.n_super_m * s.gn + p / s.gm;
  if (mt >= s.m_tiles || unit >= s.B * s.n_tiles_ub) return;
  const int b = unit / s.n_tiles_ub;
  const TokenTile tt =
      find_token_tile<kT>(s.gs + (int64_t)b * s.E, s.E, s.N, unit - b * s.n_tiles_ub);
  if (tt.e < 0) return;
  const int m0 = mt * kT;
  const int64_t ge = (int64_t)b * s.E + tt.e, row = (int64_t)b * s.N + tt.start;
  Loader<AMAJ> la;
  Loader<KMajor> lx;
  auto pair = [&](int i) __attribute__((always_inline)) {
    const int K = s.K[i];
    la.init(Operand{s.a[i] + ge * s.M * K, AMAJ == KMajor ? K : s.M, s.M, K}, m0);
    lx.init(Operand{s.x[i] + row * K, K, tt.size, K}, tt.n0);
  };
  pair(0);
  const int nk0 = (s.K[0] + kTK - 1) / kTK, nk1 = (s.K[1] + kTK - 1) / kTK;
  Acc acc;
  zero_acc(acc);
  k_loop<AMAJ, KMajor>(la, lx, nk0 + nk1, ring, acc, 1.0f,
                       [&](int k) __attribute__((always_inline)) {
                         if (k == nk0) pair(1);
                         return k < nk0 ? k : k - nk0;
                       });
  const int me = after_loop(m0), left = after_loop(tt.size) - after_loop(tt.n0);
  uint16_t* y = uniform_ptr(s.y + ((int64_t)after_loop(b) * s.N + after_loop(tt.start) +
                                   after_loop(tt.n0)) * s.M + me);
  staged(
      acc, reinterpret_cast<float*>(ring), [](auto, auto, int, int) {},
      [&](auto, auto, int n, int g, float (&v)[8]) __attribute__((always_inline)) {
        if (n < left && me + 8 * g < s.M) store8_bf16(y + (uint32_t)(n * s.M + 8 * g), v);
      });
}

// ========================================================= Newton-Schulz ==
// The three products of a step over BE matrices, with the rounding of the
// reference's bf16 tensor arithmetic, a rounding after every operation:
//   kNsA  A = bf16(X X^T).  Symmetric bit for bit: only the tiles on or below
//         the diagonal run, and one below it also stores its transpose.
//   kNsB  B = bf16(bf16(b A) + bf16((c A) A)): A's rows are both operands, the
//         second rounded to bf16(c A) as its fragments are read, so that c A
//         never goes through memory.
//   kNsX  X' = bf16(bf16(a X) + bf16(B X)); the last step stores
//         bf16(X' scale) into the caller's output, transposed for a matrix
//         with more rows than columns.
// 288 matrices of 384 x 384 read and write 85 MB per operand and product,
// which is what bounds them; 256 x 256 tiles (half padding there) took 180 / 134
// / 136 us per product.
// Every XCD takes a contiguous eighth of the tiles of all matrices: with a
// matrix per XCD, few matrices left XCDs idle (one of 4096 x 4096 12.1 ms, now
// 2.0; nine of 1536 x 3072 2.45 -> 1.82; the 256 x 256 tiles took 2.2 and 2.3).
// Within a matrix the tiles run in bands of kNsBand rows, so that the 64 on an
// XCD at once share eight rows' and eight columns' operands in its L2.
enum NsProduct { kNsA = 0, kNsB = 1, kNsX = 2 };
constexpr int kNsBand = 8;

struct Ns192Args {
  const uint16_t* a;   // per matrix: [M, K] rows, or [K, M] (kNsX)
  const uint16_t* x;   // per matrix [R, K]
  const uint16_t* in;  // per matrix [R, M] (kNsB, kNsX)
  uint16_t* y;         // per matrix [R, M], or [M, R] with `trans`
  int K, M, R, BE, m_tiles, r_tiles;
  float alpha, gamma;  // alpha: of `in`; gamma: c (kNsB), the output scale (kNsX, `last`)
  int last, trans;
};

template <int P>
__global__ __launch_bounds__(kTThreads, 2) void ns192_kernel(Ns192Args s) {
  constexpr int kAMaj = P == kNsX ? RMajor : KMajor;
  __shared__ __attribute__((aligned(16))) uint8_t ring[kTRing * kTStage];
  const int per = P == kNsA ? s.m_tiles * (s.m_tiles + 1) / 2 : s.m_tiles * s.r_tiles;
  const int unit = xcd_run(s.BE * per);
  if (unit < 0) return;
  const int mat = unit / per, t = unit % per;
  int mt, rt;
  if constexpr (P == kNsA) {  // tile t of the lower triangle, row rt holding rt + 1
    rt = 0;
    mt = t;
    while (mt > rt) mt -= ++rt;
  } else {  // bands of kNsBand rows of tiles, column by column
    const int band = t / (kNsBand * s.m_tiles) * kNsBand, p = t - band * s.m_tiles;
    const int rows = min(kNsBand, s.r_tiles - band);
    rt = band + p % rows;
    mt = p / rows;
  }
  const int m0 = mt * kT, r0 = rt * kT;
  const int64_t om = (int64_t)mat * s.R * s.M;
  const Operand A{s.a + (int64_t)mat * s.M * s.K, kAMaj == KMajor ? s.K : s.M, s.M, s.K};
  const Operand X{s.x + (int64_t)mat * s.R * s.K, s.K, s.R, s.K};
  Loader<kAMaj> la;
  Loader<KMajor> lx;
  la.init(A, m0);
  lx.init(X, r0);
  Acc acc;
  zero_acc(acc);
  k_loop<kAMaj, KMajor, P == kNsB>(la, lx, (s.K + kTK - 1) / kTK, ring, acc, s.gamma);
  // the epilogue's coordinates from opaque copies, so that no address of it is
  // held across the K loop
  const int me = after_loop(m0), re = after_loop(r0);
  // a half's `in` is loaded from clamped addresses before the half is staged
  uint4 raw[kTItems];
  const int64_t row0 = om + (int64_t)re * s.M;
  const uint16_t* in = uniform_ptr(s.in + row0);
  uint16_t* y = uniform_ptr(s.y + row0);
  uint16_t* yt = uniform_ptr(s.y + om + (int64_t)me * s.R);
  const bool trans = P == kNsX && s.trans;
  staged(
      acc, reinterpret_cast<float*>(ring),
      [&](auto, auto K, int n, int g) __attribute__((always_inline)) {
        if constexpr (P != kNsA) {
          const int r = re + n, m = me + 8 * g;
          const uint32_t at = r < s.R && m < s.M ? (uint32_t)(n * s.M + m) : 0u;
          raw[K] = *reinterpret_cast<const uint4*>(in + at);
        }
      },
      [&](auto, auto K, int n, int g, float (&v)[8]) __attribute__((always_inline)) {
        const int r = re + n, m = me + 8 * g;
        if constexpr (P != kNsA) {
          float x[8];
          unpack8_bf16(raw[K], x);
#pragma unroll
          for (int u = 0; u < 8; ++u) v[u] = bf16r(bf16r(s.alpha * x[u]) + bf16r(v[u]));
          if (P == kNsX && s.last) {
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] *= s.gamma;
          }
        }
        if (!trans && r < s.R && m < s.M) store8_bf16(y + (uint32_t)(n * s.M + m), v);
      },
      P == kNsA ? m0 != r0 : trans,
      [&](int r, int n, const float (&v)[8]) __attribute__((always_inline)) {
        if (me + r < s.M && re + n < s.R)  // R is a multiple of 8
          store8_bf16(yt + (uint32_t)(r * s.R + re + n), v);
      });
}

int tiles_of(int n) { return (n + kT - 1) / kT; }

}  // namespace

// ------------------------------------------------------------------ host ----
constexpr int kWgRuns = 64;  // runs of tiles that the weight gradients deal to the XCDs at least
Wg192Plan wg192_plan(int B, int E, int I, int D, int N) {
  Wg192Plan p{};
  // dW0_W2 [2I][D] and dW1 [D][I]
  p.per = tiles_of(2 * I) * tiles_of(D) + tiles_of(D) * tiles_of(I);
  const auto tiles_256 = [](int n) { return (int64_t)(n + 255) / 256; };
  const int64_t per256 = tiles_256(2 * I) * tiles_256(D) + tiles_256(D) * tiles_256(I);
  const int64_t tiles256 = B * E * per256;
  // tile area against that of the 256 x 256 tiles: at most 3/4, at most 1.05
  const int64_t area192 = (int64_t)p.per * kT * kT, area256 = per256 * 65536;
  const bool less = 4 * area192 <= 3 * area256, alike = 20 * area192 <= 21 * area256;
  const int64_t mean = N / std::max(E, 1);
  p.use = E > 1 && N > 0 &&
          ((less && (tiles256 > 64 || mean <= 512)) ||
           (mean <= 256 && tiles256 < 2048 &&
            (tiles256 <= 64 || (alike && (tiles256 <= 128 || tiles256 > 256)))));
  const bool narrow = I <= 512 && D <= 512;
  int chunk = narrow ? 512 : 4096;
  while (chunk < 2 * D ||
         (narrow && chunk < 4096 && (int64_t)chunk * 256 < (int64_t)B * N * p.per))
    chunk *= 2;
  p.chunk = chunk;
  p.slots = (N + chunk - 1) / chunk + E;
  p.parts_ub = N > chunk ? (int)(2 * (int64_t)N / chunk) : 0;
  p.n_out = (int64_t)3 * I * D;
  p.bytes = (size_t)B * p.parts_ub * p.n_out * sizeof(float);
  return p;
}

int launch_wg192(const Wg192Plan& pl, const void* dy, const void* k, const void* hid,
                 const void* v, void* dw0_w2, void* dw1, const int32_t* gs, int B, int E, int I,
                 int D, int N, void* workspace, hipStream_t st, const char* what) {
  const int64_t units = (int64_t)B * pl.slots;
  const int run = (int)std::max<int64_t>(1, std::min<int64_t>(pl.per, pl.per * units / kWgRuns));
  const int64_t blocks = (units * ((pl.per + run - 1) / run) + kXcds - 1) / kXcds * kXcds * run;
  UTTT_REQUIRE(blocks <= 0x7fffffffLL, "%s: problem too large for one launch", what);
  Wg192Args a{};
  auto task = [](const void* p, const void* q, void* out, int X, int Y) {
    return Wg192Task{static_cast<const uint16_t*>(p), static_cast<const uint16_t*>(q),
                     static_cast<uint16_t*>(out), X, Y, tiles_of(Y), tiles_of(X)};
  };
  a.t[0] = task(k, dy, dw0_w2, 2 * I, D);
  a.t[1] = task(hid, v, dw1, D, I);
  a.gs = gs;
  a.part = static_cast<float*>(workspace);
  a.n_out = pl.n_out;
  a.B = B;
  a.E = E;
  a.N = N;
  a.chunk = pl.chunk;
  a.slots = pl.slots;
  a.run = run;
  a.parts_ub = pl.parts_ub;
  hipLaunchKernelGGL(wg192_kernel, dim3((unsigned)blocks), dim3(kTThreads), 0, st, a);
  if (int rc = check_launch(what)) return rc;
  if (pl.parts_ub == 0) return UTTT_OK;  // no expert has a second chunk
  const int each = (int)std::min<int64_t>((pl.n_out / 8 + 255) / 256, 64);
  UTTT_REQUIRE((int64_t)B * E * each <= 0x7fffffffLL, "%s: problem too large for one launch", what);
  hipLaunchKernelGGL(wg192_reduce_kernel, dim3((unsigned)(B * E * each)), dim3(256), 0, st, a, each);
  return check_launch(what);
}

int launch_tn192(bool a_kmajor, const void* a0, const void* x0, int K0, const void* a1,
                 const void* x1, int K1, int M, void* y, int B, int E, int N, const int32_t* gs,
                 hipStream_t st, const char* what) {
  Tn192Args s{};
  s.a[0] = static_cast<const uint16_t*>(a0);
  s.x[0] = static_cast<const uint16_t*>(x0);
  s.a[1] = static_cast<const uint16_t*>(K1 > 0 ? a1 : a0);
  s.x[1] = static_cast<const uint16_t*>(K1 > 0 ? x1 : x0);
  s.K[0] = K0;
  s.K[1] = K1;
  s.y = static_cast<uint16_t*>(y);
  s.gs = gs;
  s.B = B;
  s.E = E;
  s.N = N;
  s.M = M;
  s.m_tiles = tiles_of(M);
  s.n_tiles_ub = tiles_of(N) + E;
  const int64_t units = (int64_t)B * s.n_tiles_ub;
  s.gm = std::min(s.m_tiles, 8);
  s.gn = units * s.m_tiles >= 8 * 512 ? 64 / s.gm : 1;
  s.n_super_m = (s.m_tiles + s.gm - 1) / s.gm;
  const int64_t supers = s.n_super_m * ((units + s.gn - 1) / s.gn);
  const int64_t blocks = (supers + kXcds - 1) / kXcds * kXcds * s.gm * s.gn;
  UTTT_REQUIRE(blocks <= 0x7fffffffLL && K0 < (1 << 23) && K1 < (1 << 23) && M < (1 << 23),
               "%s: problem too large for one launch", what);
  if (a_kmajor)
    hipLaunchKernelGGL((tn192_kernel<KMajor>), dim3((unsigned)blocks), dim3(kTThreads), 0, st, s);
  else
    hipLaunchKernelGGL((tn192_kernel<RMajor>), dim3((unsigned)blocks), dim3(kTThreads), 0, st, s);
  return check_launch(what);
}

namespace {
template <int P>
int launch_ns(const Ns192Args& s, hipStream_t st, const char* what) {
  const int64_t per = P == kNsA ? (int64_t)s.m_tiles * (s.m_tiles + 1) / 2
                                : (int64_t)s.m_tiles * s.r_tiles;
  const int64_t blocks = xcd_run_blocks(s.BE * per);
  UTTT_REQUIRE(blocks <= 0x7fffffffLL, "%s: problem too large for one launch", what);
  hipLaunchKernelGGL((ns192_kernel<P>), dim3((unsigned)blocks), dim3(kTThreads), 0, st, s);
  return check_launch(what);
}
}  // namespace

int launch_ns192_step(const uint16_t* x, uint16_t* a, uint16_t* b, uint16_t* xn, int BE, int m,
                      int n, float ca, float cb, float cc, bool last, float out_scale, bool trans,
                      hipStream_t st) {
  const int mt = tiles_of(m), nt = tiles_of(n);
  if (int rc = launch_ns<kNsA>({x, x, nullptr, a, n, m, m, BE, mt, mt, 0.0f, 1.0f, 0, 0}, st,
                               "newton_schulz5(X X^T)"))
    return rc;
  if (int rc = launch_ns<kNsB>({a, a, a, b, m, m, m, BE, mt, mt, cb, cc, 0, 0}, st,
                               "newton_schulz5(B)"))
    return rc;
  return launch_ns<kNsX>({x, b, x, xn, m, n, m, BE, nt, mt, ca, out_scale, last ? 1 : 0,
                          last && trans ? 1 : 0},
                         st, "newton_schulz5(B X)");
}

}  // namespace uttt
