// Decode projections of wide models (ops_wide.hip): y[m][n] = sum_k x[m][k] W[n][k] for 1..8 sequences and rows too long for the register
// and LDS images of the other decode kernels.
#pragma once

#include "engine_common.hip.h"

namespace pgk {

// where the activations come from: fp32 rows normalised on the way in, plain fp32 rows, the split pieces a SwiGLU epilogue left, and for one sequence: NORM with
// `nsplit` partial vectors added and the sum left in h_out (EPI_SWIGLU); records (m, l, o[D]) of `nsplit` slices per head of D columns, merged (EPI_STORE: out =
// wide_merge_parts(K) partial vectors)
enum { WIDE_NORM = 0, WIDE_PLAIN, WIDE_PIECES, WIDE_NORM_SUM, WIDE_MERGE };
constexpr int WIDE_RUN = 2048;                               // columns of a partial vector's product
inline int wide_merge_parts(int K) { return (K + WIDE_RUN - 1) / WIDE_RUN; }
// Every workgroup of a run reads its heads' records, 8 KB a slice and run: few slices cost less than the merge's launch (o_proj 5.6 -> 7.2 us with 12 slices, the launch 5.0, the sum of two partial
// vectors in gate_up 0.2).  Llama-3-8B shape, us a step, before / after: e4m3, contexts of 32 and 200 2151 / 2049 and 2153 / 2054, 700 2091 / 2060; bf16, 700 3040 / 2993; with 24
// slices, 1500 3057 / 3079: not beyond 16
constexpr int WIDE_SLICES = 16;
inline bool wide_merge_ok(int K, int D, int slices) { return K % 256 == 0 && (D == 64 || D == 128) && slices <= WIDE_SLICES; }

// Split pieces of M rows of K: [K / 32][M][3][4][8] bf16, three pieces each
inline size_t wide_pieces_elems(int K, int M) { return (size_t)K * M * 3; }

// x rows in registers: K <= 4096; pieces: any K; both: K % 256 == 0
bool wide_proj_ok(int N, int K, bool pieces);
// src / epi: WIDE_* and EPI_*.  Uses a.w, wscale, N, K, h (NORM) or xin (PLAIN), part, nsplit (NORM_SUM, MERGE), h_out (NORM_SUM), ld_out = D (MERGE), gamma, eps, out, ld_out (RESID: out += y), amax_val / amax_idx
// (LOGITS: *n_blk slots per row); pieces: the pieces read (WIDE_PIECES) or written (EPI_SWIGLU: for a projection of the same weight type).
pgk_status wide_proj(bool fp8, int src, int epi, const FusedArgs& a, bf16* pieces, int M, int cu_count, int* n_blk, hipStream_t st);

}  // namespace pgk
