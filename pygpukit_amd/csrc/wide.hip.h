// Decode projections of wide models (ops_wide.hip): y[m][n] = sum_k x[m][k] W[n][k] for 1..8 sequences and rows too long for the register
// and LDS images of the other decode kernels.
#pragma once

#include "engine_common.hip.h"

namespace pgk {

// where the activations come from: fp32 rows normalised on the way in, plain fp32 rows, or the split pieces a SwiGLU epilogue left
enum { WIDE_NORM = 0, WIDE_PLAIN, WIDE_PIECES };

// Split pieces of M rows of K: [K / 32][M][3][4][8] bf16, three pieces each
inline size_t wide_pieces_elems(int K, int M) { return (size_t)K * M * 3; }

// x rows in registers: K <= 4096; pieces: any K; both: K % 256 == 0
bool wide_proj_ok(int N, int K, bool pieces);
// src / epi: WIDE_* and EPI_*.  Uses a.w, wscale, N, K, h (NORM) or xin (PLAIN), gamma, eps, out, ld_out (RESID: out += y), amax_val / amax_idx
// (LOGITS: *n_blk slots per row); pieces: the pieces read (WIDE_PIECES) or written (EPI_SWIGLU: for a projection of the same weight type).
pgk_status wide_proj(bool fp8, int src, int epi, const FusedArgs& a, bf16* pieces, int M, int cu_count, int* n_blk, hipStream_t st);

}  // namespace pgk
