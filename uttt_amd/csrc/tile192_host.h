// Host side of the 192 x 192 tile kernels (tile192.hip).
#pragma once

#include "common.h"

namespace uttt {

// Chunked weight gradients of the grouped UPDATE on 192 x 192 tiles: `use`
// where they are the faster ones, a pure function of the sizes (so the
// workspace query and the launch agree), from 3000 sizes (2 to 128 experts, I
// and D from 64 to 512 and wider with short segments, 64 to 196 608 tokens) timed on
// both:
//   - at most 3/4 of the 256 x 256 tiles' area (sides of 192, 320, 384): 48
//     experts of 192 x 192 over 196 608 tokens 285-459 -> 105 us; 96 of 384 x
//     384 over 16 384 70 -> 46, over 196 608 374 -> 290.  Not with few tiles and
//     long segments, which the split-K 256 tiles cover (4 experts of 192 x 384
//     over 4096 tokens 19 / 23 us);
//   - means of at most 256 tokens, where a prologue and an epilogue per tile
//     weigh most: with few tiles any width, else a like area (16 experts of 768
//     x 1536 over 3062 tokens 71 -> 57 us), but not in place of one even round
//     of 256 tiles on the 256 CUs (32 of 64 x 512 over 8192 27 / 32 us).
// Sides of 256 and 512 pad by up to 1.9 times (8 experts of 512 x 256 over
// 196 608 tokens 196 / 374 us).  One expert per batch (uTTT-Dense heads): the
// split-K 256 tiles measure the same or faster (4 x [192 x 384] over 98 304
// tokens 79 / 90 us).  Still up to 1.3 times slower: 8 to 32 experts, or 16 batches
// of 4, with long segments of one length (32 of 384 x 192 over 98 304: 83 / 109 us),
// where unequal ones are up to twice faster.
// Chunk length: about 256 (chunk, tile) workgroups on an even routing, 512 to
// 4096 tokens (4096 with a side above 512), at least 2 D: a batch's partials then
// fit in the backward's dead intermediates, 12 N I bytes.
struct Wg192Plan {
  bool use;
  int per;        // output tiles of one expert
  int chunk;      // tokens per chunk
  int slots;      // upper bound of the chunks of one batch
  int parts_ub;   // upper bound of its partial chunks
  int64_t n_out;  // output elements of one expert
  size_t bytes;   // fp32 partials
};
Wg192Plan wg192_plan(int B, int E, int I, int D, int N);

// dW0_W2 [2I][D] = DY^T K and dW1 [D][I] = V^T Hid of every expert.  I, D
// multiples of 8, pointers 16-byte aligned; `workspace` holds plan.bytes.
int launch_wg192(const Wg192Plan& plan, const void* dy, const void* k, const void* hid,
                 const void* v, void* dw0_w2, void* dw1, const int32_t* gs, int B, int E, int I,
                 int D, int N, void* workspace, hipStream_t st, const char* what);

// Token-grouped products y[b, n, m] = sum_k A(m, k) x[b, n, k], a second pair
// chained along k when K1 > 0.  Widths multiples of 8, pointers 16-byte aligned.
int launch_tn192(bool a_kmajor, const void* a0, const void* x0, int K0, const void* a1,
                 const void* x1, int K1, int M, void* y, int B, int E, int N, const int32_t* gs,
                 hipStream_t st, const char* what);

// One Newton-Schulz step of BE matrices x [m, n] (m <= n): a [m, m] = x x^T,
// b [m, m] = cb a + (cc a) a, xn [m, n] = ca x + b x; `last`: xn times
// out_scale, as [n, m] with `trans`.
int launch_ns192_step(const uint16_t* x, uint16_t* a, uint16_t* b, uint16_t* xn, int BE, int m,
                      int n, float ca, float cb, float cc, bool last, float out_scale, bool trans,
                      hipStream_t st);

}  // namespace uttt
