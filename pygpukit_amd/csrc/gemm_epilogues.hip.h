// Arguments of the GEMM epilogues that finish an engine step inside the projection (ops_gemm256.hip; callers: ops_gemm.hip, engine.hip).
#pragma once
#include "pgk_device.hip.h"

namespace pgk {

// QKV projection whose tile columns are whole heads (head_dim 128): per (token row, head slot) the bf16-rounded result gets the
// per-head RMSNorm (q / k heads, when a gamma is given) and RoPE; q heads are stored to the qkv buffer, k / v heads to the KV
// cache row of the token's position - what qknorm_rope_kvwrite_kernel (engine.hip) does in a pass of its own.
struct QkvHeadArgs {
    const bf16 *q_gamma, *k_gamma;        // null: no per-head norm
    float eps;
    const float *rope_cos, *rope_sin;     // [max_seq][64]
    bf16 *kcache, *vcache;                // this layer's, this sequence's: [Hkv][max_seq][128]
    int hq, hkv, max_seq, start_pos;
    // rows of several sequences: (position, slot) of each; kcache / vcache are then slot 0's and slot_stride elements apart.  Null: position
    // start_pos + row
    const int2* at;
    long long slot_stride;
};
// An RMSNorm between two products without a pass of its own.  The product before it (its residual epilogue) leaves x = bf16(h gamma) and, per row and 64
// columns, h's sum of squares; the product behind it reads x and scales its result rows by 1 / rms, which a factor per row may as well do after the sum.
// ss [n][rows], or (ld = 64) [rows][64] of which n <= 64 count, as pkgemm_resid_nt leaves them; null: x is normalised
struct NormIn { const float* ss; int n; float eps; int ld; };
struct NormOut { const bf16* gamma; bf16* x; float* ss; };  
// 1 / rms of a row of K values
__device__ __forceinline__ float norm_in_scale(const NormIn& nn, int row, int rows, int K) {
    float s = 0.f;
    for (int i = 0; i < nn.n; i += 16) {
        float v[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) v[j] = nn.ss[(size_t)min(i + j, nn.n - 1) * rows + row];
#pragma unroll
        for (int j = 0; j < 16; ++j) s += i + j < nn.n ? v[j] : 0.f;
    }
    return 1.0f / sqrtf(s / K + nn.eps);
}
// Residual epilogue of four columns of a row (gamma: g), held by one of 16 lanes that have 64: h (already stored) -> x and the sum of squares.  All lanes must be active.
__device__ __forceinline__ void norm_out_row(const float4& v, uint2 g, bool live, int row, int col, int rows, int N, const NormOut& no) {
    const float ss = group16_sum(live ? v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w : 0.f);
    if (!live) return;
    uint2 o;
    o.x = pack_bf16x2(v.x * __uint_as_float(g.x << 16), v.y * __uint_as_float(g.x & 0xFFFF0000u));
    o.y = pack_bf16x2(v.z * __uint_as_float(g.y << 16), v.w * __uint_as_float(g.y & 0xFFFF0000u));
    *reinterpret_cast<uint2*>(no.x + (size_t)row * N + col) = o;
    if ((col & 63) == 0) no.ss[(size_t)(col >> 6) * rows + row] = ss;
}
struct ActArgs { float pos, neg; bool gelu; };     // pgk_device.hip.h: xielu's factors, or gelu_erf

// Head slots of the bf16-rounded QKV projection of ROWS token rows, row0 + step i: 16 lanes hold one row's 128 dims, 8 each (sub = lane's chunk).
// finish() does the arithmetic of qknorm_rope_kvwrite_kernel, operation for operation, then the store (load(i) gives a row's dims); all lanes must be active.
// The rows' places and angles are asked for by places() and angles(), which callers put ahead of and behind the writes of the tile to LDS: two round trips that
// the tile's barrier hides.  Asked for four rows at a time between the stores, the epilogue of a 256-row tile (two heads) took 9.9 us of the 32 of a product of
// 3365 x 4096 x 1024, and 4.3 of 14 for a 128-row tile.
template <int ROWS>
struct HeadRows {
    int2 place[ROWS];
    float4 cs[ROWS][2], sn[ROWS][2];
    __device__ __forceinline__ void places(int row0, int step, int M, const QkvHeadArgs& hd) {
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
            const int grow = row0 + i * step;
            place[i] = hd.at ? hd.at[min(grow, M - 1)] : make_int2(hd.start_pos + grow, 0);
        }
    }
    __device__ __forceinline__ void angles(int sub, int first_slot, const QkvHeadArgs& hd) {
        if (first_slot >= hd.hq + hd.hkv) return;            // value heads are stored as they are
        const int dd = (sub * 8) % 64;
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
            const size_t at = (size_t)min(place[i].x, hd.max_seq - 1) * 64 + dd;
            cs[i][0] = *reinterpret_cast<const float4*>(hd.rope_cos + at); cs[i][1] = *reinterpret_cast<const float4*>(hd.rope_cos + at + 4);
            sn[i][0] = *reinterpret_cast<const float4*>(hd.rope_sin + at); sn[i][1] = *reinterpret_cast<const float4*>(hd.rope_sin + at + 4);
        }
    }
    template <class Load>
    __device__ __forceinline__ void finish(int sub, int slot, int row0, int step, int M, const QkvHeadArgs& hd, bf16* qkv, int ldq, Load load) const {
        const bool is_q = slot < hd.hq, is_k = !is_q && slot < hd.hq + hd.hkv;
        const bf16* gamma = is_q ? hd.q_gamma : hd.k_gamma;
        Vec<bf16> gr;
        gr.raw = make_uint4(0, 0, 0, 0);
        if (gamma) gr.raw = *reinterpret_cast<const uint4*>(gamma + sub * 8);
        float gm[8];
        gr.to_float(gm);
        const float sign = sub < 8 ? -1.f : 1.f;
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
            const int grow = row0 + i * step, pos = place[i].x;
            float x[8];
            load(i, x);
            if (is_q || is_k) {
                if (gamma) {
                    float ss = 0.f;
#pragma unroll
                    for (int j = 0; j < 8; ++j) ss = fmaf(x[j], x[j], ss);
                    ss = group_sum<16>(ss);
                    const float inv = 1.0f / sqrtf(ss / 128 + hd.eps);
#pragma unroll
                    for (int j = 0; j < 8; ++j) x[j] = x[j] * inv * gm[j];
                }
                const float c[8] = {cs[i][0].x, cs[i][0].y, cs[i][0].z, cs[i][0].w, cs[i][1].x, cs[i][1].y, cs[i][1].z, cs[i][1].w};
                const float s[8] = {sn[i][0].x, sn[i][0].y, sn[i][0].z, sn[i][0].w, sn[i][1].x, sn[i][1].y, sn[i][1].z, sn[i][1].w};
                float o[8];
                // x c -+ other s
#pragma unroll
                for (int j = 0; j < 8; ++j) o[j] = fmaf(x[j], c[j], xor_half<16>(x[j]) * (s[j] * sign));
#pragma unroll
                for (int j = 0; j < 8; ++j) x[j] = o[j];
            }
            Vec<bf16> ov;
            ov.from_float(x);
            if (grow < M) {
                if (is_q) {
                    ov.store(qkv + (size_t)grow * ldq + slot * 128 + sub * 8);
                } else if (pos < hd.max_seq) {
                    const int kvh = is_k ? slot - hd.hq : slot - hd.hq - hd.hkv;
                    ov.store((is_k ? hd.kcache : hd.vcache) + place[i].y * hd.slot_stride + ((size_t)kvh * hd.max_seq + pos) * 128 + sub * 8);
                }
            }
        }
    }
};

}  // namespace pgk
