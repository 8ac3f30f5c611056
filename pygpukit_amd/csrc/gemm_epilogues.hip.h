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
struct ActArgs { float pos, neg; bool gelu; };     // pgk_device.hip.h: xielu's factors, or gelu_erf

// Head slot `slot` of the bf16-rounded QKV projection of ROWS token rows, row0 + STEP i: 16 lanes hold one row's 128 dims, 8 each (sub = lane's
// chunk; load(i) gives them).  The arithmetic of qknorm_rope_kvwrite_kernel, operation for operation, then the store.  All lanes must be active.
// Four rows' places and angles are requested together, ahead of the stores, which the compiler cannot move them across: a row at a time the
// epilogue was a chain of ROWS round trips (QKV of Qwen3-0.6B, 3365 rows in 256-tiles 45 -> 42 us, 384 rows in 128-tiles 16.9 -> 15.2).
template <int ROWS, int STEP, class Load>
__device__ __forceinline__ void qkv_heads_finish(int sub, int slot, int row0, int M, const QkvHeadArgs& hd, bf16* qkv, int ldq, Load load) {
    const bool is_q = slot < hd.hq, is_k = !is_q && slot < hd.hq + hd.hkv;
    const bf16* gamma = is_q ? hd.q_gamma : hd.k_gamma;
    Vec<bf16> gr;
    gr.raw = make_uint4(0, 0, 0, 0);
    if (gamma) gr.raw = *reinterpret_cast<const uint4*>(gamma + sub * 8);
    float gm[8];
    gr.to_float(gm);
    const int dd = (sub * 8) % 64;
    const bool lo = sub < 8;
#pragma unroll
    for (int i0 = 0; i0 < ROWS; i0 += 4) {
        int2 place[4];
        float4 cs[4][2], sn[4][2];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int grow = row0 + (i0 + u) * STEP;
            place[u] = hd.at ? hd.at[min(grow, M - 1)] : make_int2(hd.start_pos + grow, 0);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const size_t at = (size_t)min(place[u].x, hd.max_seq - 1) * 64 + dd;
            cs[u][0] = *reinterpret_cast<const float4*>(hd.rope_cos + at); cs[u][1] = *reinterpret_cast<const float4*>(hd.rope_cos + at + 4);
            sn[u][0] = *reinterpret_cast<const float4*>(hd.rope_sin + at); sn[u][1] = *reinterpret_cast<const float4*>(hd.rope_sin + at + 4);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int grow = row0 + (i0 + u) * STEP, pos = place[u].x;
            float x[8];
            load(i0 + u, x);
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
                const float c[8] = {cs[u][0].x, cs[u][0].y, cs[u][0].z, cs[u][0].w, cs[u][1].x, cs[u][1].y, cs[u][1].z, cs[u][1].w};
                const float s[8] = {sn[u][0].x, sn[u][0].y, sn[u][0].z, sn[u][0].w, sn[u][1].x, sn[u][1].y, sn[u][1].z, sn[u][1].w};
                float o[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const float other = xor_half<16>(x[j]);
                    o[j] = lo ? (x[j] * c[j] - other * s[j]) : (x[j] * c[j] + other * s[j]);
                }
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
                    ov.store((is_k ? hd.kcache : hd.vcache) + place[u].y * hd.slot_stride + ((size_t)kvh * hd.max_seq + pos) * 128 + sub * 8);
                }
            }
        }
    }
}

}  // namespace pgk
