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
// output rows of a workgroup where `runs` runs of columns share the CUs: one workgroup each
inline int wide_rows(int N, int cu_count, int runs) { return ceil_div(ceil_div(N, runs < cu_count ? cu_count / runs : 1), 8) * 8; }
constexpr int WIDE_SLICES = 16;
inline bool wide_merge_ok(int K, int D, int slices) { return K % 256 == 0 && (D == 64 || D == 128) && slices <= WIDE_SLICES; }
// Every workgroup of a run reads its heads' records, 8 KB a slice and run: few slices cost less than the merge's launch (e4m3, 12 slices, o_proj 5.6 -> 7.5 us, the launch 5.0, the sum of two partial
// vectors in gate_up 0.2).  Llama-3-8B shape, e4m3, us a step, before / after: contexts of 32 and 200 2151 / 2049 and 2153 / 2054, 700 2091 / 2060; with 24 slices even: not beyond 16.
// Nor where the weights that wait behind the records are more than 64 KB a workgroup, as bf16 ones of width 2560 and more are with two runs: o_proj 7.7 -> 11.2 us there.  8 layers, bf16, us a step,
// with the launch / without: width 4096, 12 slices 747 / 755, 16 slices 772 / 784, of 32 kv heads 735 / 743; 3072 511 / 515; 2560 506 / 513; but 2048, 4096 columns 422 / 415, 1536, 2304 columns 357 / 344.
inline bool wide_merge_pays(bool fp8, int N, int K, int cu_count) {
    return (size_t)wide_rows(N, cu_count, wide_merge_parts(K)) * (K < WIDE_RUN ? K : WIDE_RUN) * (fp8 ? 1 : 2) <= 64 * 1024;
}

// Split pieces of M rows of K: [K / 32][M][3][4][8] bf16, three pieces each
inline size_t wide_pieces_elems(int K, int M) { return (size_t)K * M * 3; }

// x rows in registers: K <= 4096; pieces: any K; both: K % 256 == 0
bool wide_proj_ok(int N, int K, bool pieces);
// src / epi: WIDE_* and EPI_*.  Uses a.w, wscale, N, K, h (NORM) or xin (PLAIN), part, nsplit (NORM_SUM, MERGE), h_out (NORM_SUM), ld_out = D (MERGE), gamma, eps, out, ld_out (RESID: out += y), amax_val / amax_idx
// (LOGITS: *n_blk slots per row); pieces: the pieces read (WIDE_PIECES) or written (EPI_SWIGLU: for a projection of the same weight type).
pgk_status wide_proj(bool fp8, int src, int epi, const FusedArgs& a, bf16* pieces, int M, int cu_count, int* n_blk, hipStream_t st);

}  // namespace pgk
