// Host side of the narrow-expert UPDATE kernels (narrow.hip).
#pragma once

#include "common.h"

namespace uttt {

// Expert widths that narrow.hip's kernels take (any token counts).
bool narrow_experts(int I, int D);
// Sizes whose stage 1 it takes: also experts up to 768 x 1536 elements (the
// product: 288 x 4096 and 4096 x 288 gain alike) with at most 256 tokens on
// average, where half of the 256-token tiles is padding and the fp32 DH a round
// trip (16 over 3062 tokens: DH 34 + 64 us, here 69).  Past 128 tokens only with
// all weights within the 256 MB memory-side cache, since a second 128-token tile
// then reads them again (128 experts of 768 x 1536 over 20 480: 333 / 405 us).
// Their backward gains nothing (GD 24 + 67 us, here 93 and twice the lr
// partials).  Of 3600 timings (1 to 128 experts, widths 8 to 8192) none is over
// 6 % slower than the two launches, and of as many gate/up ones one (a few tokens
// per expert, 9.6 / 10.5 us).
bool narrow_stage1(int I, int D, int N, int B, int E);
// Whose backward it takes: those widths, but not many tokens of experts that fill
// both of the general tiles' 256s, which reuse a token's row for twice the units
// (timings of 7 widths from 384 x 512; 16 experts of 480 x 512 over 131 072 tokens:
// 1288 / 1167 us here / there; 448 x 512 over 65 536 alike; 512 x 384 over 196 608
// 1604 / 1631; 512 x 512 over 16 384: 208 / 219).
bool narrow_bwd(int I, int D, int N, int B);
// Row blocks of its lr-gradient partials, lr_part[3][narrow_m_tiles][B][N].
int narrow_m_tiles(int I);

// Stage 1 with token-major outputs (uttt_grouped_update_stage1) without the
// fp32 workspace; lr0 .. lr2 and the saves may be null.
int launch_narrow_stage1(const void* w0_w2, const void* w1, const void* k, const void* v,
                         const void* lr0, const void* lr1, const void* lr2, int lr_dtype,
                         const int32_t* gs, int B, int E, int I, int D, int N, void* dy, void* hid,
                         void* y_save, void* dh_save, hipStream_t st, const char* what);

// The APPLY's gate/up, hidden [B, N, I] = silu(w0 x) * (w2 x); src_rows (rows of
// src_sb entries, or null): row n of batch b is row src_rows[b][n] of x [B, T, D].
int launch_narrow_gate_up(const void* w0_w2, const void* x, const int32_t* src_rows,
                          long long src_sb, const int32_t* gs, int B, int E, int I, int D, int N,
                          int T, void* hidden, hipStream_t st, const char* what);

// The backward's second-order pass from the saved values: grad_dh [B, N, I],
// grad_x0_x2 and dx0_x2 [B, N, 2I], hidden_lr1 [B, N, I], lr-gradient partials.
int launch_narrow_bwd(const void* gw0_w2, const void* gw1, const void* k, const void* v,
                      const void* lr0, const void* lr1, const void* lr2, int lr_dtype,
                      const int32_t* gs, int B, int E, int I, int D, int N, const void* y_saved,
                      const void* dh_saved, uint16_t* gdh, uint16_t* gx, uint16_t* dx,
                      uint16_t* hlr, float* lr_part, hipStream_t st, const char* what);

}  // namespace uttt
