// Batched decode projections on MFMA (3 <= M <= 64 sequences per launch), included by engine_batched.hip.
//
// The GEMV kernels of engine.hip score every weight chunk against M activation rows with VALU dot products: 32 packed
// dot instructions per 16-byte weight chunk at M = 8, and the kernel turns instruction-bound (gate_up 9.3 us, lm_head
// 86 us at M = 8 against 5.7 / 50 us at M = 1).  Here the M rows are the (zero-padded) A operand of
// v_mfma_f32_16x16x32_bf16 and 16 weight rows are its B operand, loaded straight from HBM in fragment shape
// (lane l: W[n0 + (l&15)][k + 8*(l>>4) ..+8], the layout of ops_wsgemm.hip): one MFMA replaces those 32 instructions and
// the cost of a projection no longer depends on M.
//   workgroup = 4 waves = 16 output rows (SWIGLU: 16 gate rows and their 16 up rows); the waves split K four ways, partial
//   16x16 tiles are summed through LDS; prologue = RMSNorm (or plain copy) of the M rows into an LDS image laid out
//   [k/8][MP] x 16 B so that an A-fragment read is 64 consecutive 16-byte slots; epilogues as in engine.hip
//   (store / residual add / SiLU(g)*u / logits + per-workgroup argmax partials, lowest index on ties).
// fp8 weights: 8 codes per lane per step, widened to bf16 with the block scale in registers (as ops_wsgemm.hip).

// Any K = 128 steps that the register-fragment kernels below do not take, up to what the image holds.  MP: activation rows held in LDS (8 or 16).
template <class WT, int PRO, int EPI, int MP>
__global__ __launch_bounds__(256) void batched_mfma_kernel(unsigned long long* tl, FusedArgs a, int M, int steps /* K / 128 per wave */, int nblk_logits) {
    const TLStamp tls(tl);
    constexpr bool FP8 = std::is_same<WT, fp8e4m3>::value;
    constexpr int NT = (EPI == EPI_SWIGLU) ? 2 : 1;       // weight row groups per workgroup
    extern __shared__ __attribute__((aligned(16))) char smem[];   // x image [K/8][MP] x 16 B | partial tiles
    __shared__ float s_ss[4][16];
    const int K = a.K, N = a.N;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, q = lane >> 4, l15 = lane & 15;
    const int ngroups = (N + 15) >> 4;                     // 16-row groups; a workgroup takes groups blockIdx.x, + gridDim.x, ...
    const int kw0 = wid * steps * 32;                      // first k of this wave
    const int em = tid >> 4, en = tid & 15;                // epilogue element of this thread: (row em, column n0 + en)

    // ---- prologue: M rows -> bf16 LDS image, chunk c (8 k) of row m at (c * MP + m) * 16 ----
    // Rows are unrolled to MP with clamped addresses and masked use (a runtime row loop would index registers
    // dynamically and wait per load); chunk loops have a uniform trip count for the same reason.
    const int nchunk = K >> 3;
    const float* src = a.h;
    if constexpr (PRO == PRO_NORM) {
        float ss[MP];
#pragma unroll
        for (int m = 0; m < MP; ++m) ss[m] = 0.f;
        for (int c0 = 0; c0 < nchunk; c0 += 256) {
            const int c = min(c0 + tid, nchunk - 1);
            const bool live = c0 + tid < nchunk;
            float4 v0[MP], v1[MP];
#pragma unroll
            for (int m = 0; m < MP; ++m) {
                v0[m] = *reinterpret_cast<const float4*>(src + (size_t)min(m, M - 1) * K + c * 8);
                v1[m] = *reinterpret_cast<const float4*>(src + (size_t)min(m, M - 1) * K + c * 8 + 4);
            }
#pragma unroll
            for (int m = 0; m < MP; ++m) {
                const float p = v0[m].x * v0[m].x + v0[m].y * v0[m].y + v0[m].z * v0[m].z + v0[m].w * v0[m].w + v1[m].x * v1[m].x +
                                v1[m].y * v1[m].y + v1[m].z * v1[m].z + v1[m].w * v1[m].w;
                ss[m] += live ? p : 0.f;
            }
        }
#pragma unroll
        for (int m = 0; m < MP; ++m) {
            const float t = wave_sum(ss[m]);
            if (lane == 0) s_ss[wid][m] = t;
        }
        __syncthreads();
    }
    for (int c0 = 0; c0 < nchunk; c0 += 256) {
        const int c = min(c0 + tid, nchunk - 1);
        if constexpr (PRO == PRO_NORM) {
            Vec<bf16> gr;
            gr.load(a.gamma + c * 8);
            float g[8];
            gr.to_float(g);
            float4 v0[MP], v1[MP];
#pragma unroll
            for (int m = 0; m < MP; ++m) {
                v0[m] = *reinterpret_cast<const float4*>(src + (size_t)min(m, M - 1) * K + c * 8);
                v1[m] = *reinterpret_cast<const float4*>(src + (size_t)min(m, M - 1) * K + c * 8 + 4);
            }
#pragma unroll
            for (int m = 0; m < MP; ++m) {
                float f[8] = {v0[m].x, v0[m].y, v0[m].z, v0[m].w, v1[m].x, v1[m].y, v1[m].z, v1[m].w};
                const float inv = 1.0f / sqrtf((s_ss[0][m] + s_ss[1][m] + s_ss[2][m] + s_ss[3][m]) / K + a.eps);
#pragma unroll
                for (int j = 0; j < 8; ++j) f[j] = f[j] * inv * g[j];
                Vec<bf16> o;
                o.from_float(f);
                if (m >= M) o.raw = make_uint4(0, 0, 0, 0);     // unused rows of the image are zero
                *reinterpret_cast<uint4*>(smem + ((size_t)c * MP + m) * 16) = o.raw;   // (duplicate writes of the clamped tail chunk are identical)
            }
        } else {                                            // bf16 hand-off: copy the stored chunks into the image
#pragma unroll
            for (int m = 0; m < MP; ++m) {
                uint4 raw = *reinterpret_cast<const uint4*>(a.xin16 + (size_t)min(m, M - 1) * K + c * 8);
                if (m >= M) raw = make_uint4(0, 0, 0, 0);
                *reinterpret_cast<uint4*>(smem + ((size_t)c * MP + m) * 16) = raw;
            }
        }
    }
    __syncthreads();

    // ---- body: one 16-row group per trip; the LDS image of the activations stays, the partial tiles have their own area ----
    float* red = reinterpret_cast<float*>(smem + (size_t)nchunk * MP * 16);   // [NT][4 waves][16 m][16 n]
    const int am = l15 & (MP - 1);
    float bv = -INFINITY;          // EPI_LOGITS: best of this thread's elements over the workgroup's groups
    int bi = 0x7FFFFFFF;
    for (int g = blockIdx.x; g < ngroups; g += gridDim.x) {
        const int n0 = g * 16;
        float resv = 0.f;
        if constexpr (EPI == EPI_RESID) resv = a.res[(size_t)min(em, M - 1) * a.ld_out + min(n0 + en, N - 1)];
        f32x4_b acc[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = f32x4_b{0.f, 0.f, 0.f, 0.f};
        for (int s = 0; s < steps; ++s) {
            const int k = kw0 + s * 32 + 8 * q;
            const uint4 af = *reinterpret_cast<const uint4*>(smem + ((size_t)((k >> 3)) * MP + am) * 16);
            const int nrow = min(n0 + l15, N - 1);
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const size_t row = (size_t)(t == 0 ? nrow : N + nrow);
                uint4 b;
                if constexpr (FP8) {
                    const uint2 v = *reinterpret_cast<const uint2*>(reinterpret_cast<const uint8_t*>(a.w) + row * K + k);
                    const float sc = to_f(a.wscale[(row >> 7) * (size_t)(K >> 7) + (k >> 7)]);
                    const f32x2 c0 = __builtin_amdgcn_cvt_pk_f32_fp8((int)v.x, false), c1 = __builtin_amdgcn_cvt_pk_f32_fp8((int)v.x, true);
                    const f32x2 c2 = __builtin_amdgcn_cvt_pk_f32_fp8((int)v.y, false), c3 = __builtin_amdgcn_cvt_pk_f32_fp8((int)v.y, true);
                    b = make_uint4(pack_bf16x2(c0.x * sc, c0.y * sc), pack_bf16x2(c1.x * sc, c1.y * sc), pack_bf16x2(c2.x * sc, c2.y * sc),
                                   pack_bf16x2(c3.x * sc, c3.y * sc));
                } else {
                    b = load_nt16(reinterpret_cast<const bf16*>(a.w) + row * K + k);
                }
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_b, af), __builtin_bit_cast(bf16x8_b, b), acc[t], 0, 0, 0);
            }
        }
        // sum the four K quarters: C tile element (m = 4 q + r, n = l15)
        __syncthreads();                                    // the previous trip's partial tiles have been read
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) red[((t * 4 + wid) * 16 + q * 4 + r) * 16 + l15] = acc[t][r];
        __syncthreads();
        float y[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const float* p = red + (size_t)t * 4 * 256 + em * 16 + en;
            y[t] = p[0] + p[256] + p[512] + p[768];
        }
        const bool ok = em < M && n0 + en < N;
        const size_t o = (size_t)em * a.ld_out + n0 + en;
        if constexpr (EPI == EPI_STORE) {
            if (ok) a.out[o] = y[0];
        } else if constexpr (EPI == EPI_RESID) {
            if (ok) a.out[o] = resv + y[0];
        } else if constexpr (EPI == EPI_SWIGLU) {
            if (ok) {
                const float act = y[0] / (1.0f + __expf(-y[0])) * y[NT - 1];
                if (a.out16) a.out16[o] = from_f<bf16>(act);
                else a.out[o] = act;
            }
        } else {   // EPI_LOGITS
            if (ok) {
                a.out[o] = y[0];
                if (y[0] > bv) { bv = y[0]; bi = n0 + en; }     // groups ascend: a later equal value never replaces an earlier one
            }
        }
    }
    if constexpr (EPI == EPI_LOGITS) {   // best of this workgroup's columns per row (lowest index on ties)
#pragma unroll
        for (int off = 8; off >= 1; off >>= 1) {
            const float ov = __shfl_xor(bv, off, 64);
            const int oi = __shfl_xor(bi, off, 64);
            if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
        }
        if (en == 0 && em < M) {
            a.amax_val[(size_t)em * nblk_logits + blockIdx.x] = bv;
            a.amax_idx[(size_t)em * nblk_logits + blockIdx.x] = bi;
        }
    }
    tls.end();
}

// ---------------------------------------------------------------------------------------------------------------------
// Register-resident variant (K = 128 S, S in {8, 16, 24, 32}): the default.
//
// The LDS-image kernel above spends its time before the first MFMA: every workgroup reads all M rows twice (sum of
// squares, then normalise), writes a K x 16 image to LDS and crosses two barriers - 9-13 us per projection at M = 16
// where the M = 1 GEMV kernels take 4.6-5.8.  A wave only ever multiplies ITS quarter of K, so here each wave takes that
// quarter of the activation rows: raw fp32 values in registers while the row sums of squares cross the waves (64 floats of LDS,
// one barrier), then bf16 through LDS of its own into A fragments: one pass over the rows, no other barrier.
// The rows are loaded along K, 1 KiB contiguous per wave instruction.  Loaded in fragment shape (lane l: row l & 15, k = 32 s + 8 (l >> 4) .. + 8) an instruction
// is 64 pieces of 16 bytes, which a CU's texture path takes at one a clock: S = 24 kept it busy for 2.8 us of a 5.5 us launch.  Us a launch of 5 rows, then and now: QKV
// (N = 4096, K = 1024) 4.0 / 2.6, o_proj (1024, 2048) 3.4 / 2.5, gate_up (6144, 1024) 4.6 / 3.4, down (1024, 3072) 4.3 / 2.8; a step of Qwen3-0.6B at contexts to 300, us: 3
// sequences 815 / 692, 8 893 / 723, 9 912 / 786, 16 1013 / 843, with e4m3 weights 8 1016 / 743; 8 layers of K = 4096 1111 / 565.
// RPG = weight rows per workgroup (16, 8 or 4): the N = hidden projections have only N / 16 = 64 row groups at
// N = 1024, far too few workgroups to pull HBM bandwidth; with RPG < 16 the lanes of the unused B columns load nothing
// and the epilogue ignores those columns (the MFMA computes them on whatever the registers hold - columns are
// independent).  MR = rows that are loaded, 8 or 16: those past the batch repeat its last one, and their results are dropped.
template <class WT, int PRO, int EPI, int S, int RPG, int MR>
__global__ __launch_bounds__(256) void batched_reg_kernel(unsigned long long* tl, const void* w_, const bf16* wp_, const float* x_, const bf16* gamma_,
                                                          int N_, int K_, int M, int nblk_logits, FusedArgs a) {
    // the first 14 dwords of the arguments - everything the load-issue phase needs - arrive preloaded in SGPRs (see fused_gemv_kernel,
    // engine.hip): w_ / wp_ = FusedArgs::w / wp, x_ = the input rows (fp32 h for the norm prologue, else xin16), gamma_, N_, K_
    const TLStamp tls(tl);
    constexpr bool FP8 = std::is_same<WT, fp8e4m3>::value;
    constexpr int NT = (EPI == EPI_SWIGLU) ? 2 : 1;
    constexpr int NC = S / 8;                              // chunks of 256 k of a wave's quarter
    static_assert(S % 8 == 0 && (MR == 8 || MR == 16), "whole chunks; 8 or 16 rows");
    __shared__ __attribute__((aligned(16))) float s_ss[MR][20];        // sums of squares: of 16 lanes of a wave, 16 parts a row
    __shared__ float red[NT * 4 * 256];                    // [NT][4 waves][16 m][16 n]
    __shared__ __attribute__((aligned(16))) char s_img[4][MR * 512];   // a wave's chunk: 8 k of row m at slot m ^ (k / 8) of MR
    const int K = K_, N = N_;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, q = lane >> 4, l15 = lane & 15;
    const int ngroups = (N + RPG - 1) / RPG;
    const int kw0 = wid * S * 32;
    // Weights of a group, every load unconditional (one under a branch is waited for where the branches meet again, in front of the whole prologue).
    // 16 rows: in fragment shape, a step (e4m3: two, a lane's 16 bytes are 8 k of each, so that a load takes 64 bytes of a row; the activations follow) to a load -
    // of the fragment-major copy (ops_pkgemm.hip: block (n-tile, k-step) is this very fragment, 1 KiB in lane order) where there is one.
    // Fewer: along K like the activations, and through the wave's LDS.
    constexpr bool FRAG = RPG == 16;
    constexpr int RL = FP8 ? 4 : 2;                        // rows of a chunk to a load
    constexpr int WS = FRAG ? (FP8 ? S / 2 : S) : NC * RPG / RL;
    uint4 wv[NT][WS];
    float wsc[NT][FRAG ? WS : NC * 2];                     // e4m3 block scales: of a load; of a half chunk of this lane's column
    auto load_w = [&](int n0) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            auto row_of = [&](int r) { return (size_t)(t == 0 ? 0 : N) + min(n0 + r, N - 1); };
            if constexpr (FRAG && !FP8) {
                const bool pk = wp_ != nullptr && n0 + 16 <= N;
                const bf16* p = pk ? wp_ + (((size_t)((t == 0 ? n0 : N + n0) >> 4) * (K >> 5) + (kw0 >> 5)) * 64 + lane) * 8
                                   : reinterpret_cast<const bf16*>(w_) + row_of(l15) * K + kw0 + 8 * q;
                const size_t step = pk ? 512 : 32;
#pragma unroll
                for (int s = 0; s < S; ++s) wv[t][s] = load_nt16(p + (size_t)s * step);
            } else if constexpr (FRAG) {
                const size_t row = row_of(l15);
#pragma unroll
                for (int s = 0; s < WS; ++s) {
                    const int k = kw0 + s * 64 + 16 * q;
                    wv[t][s] = load_nt16(reinterpret_cast<const uint8_t*>(w_) + row * K + k);
                    wsc[t][s] = to_f(a.wscale[(row >> 7) * (size_t)(K >> 7) + (k >> 7)]);
                }
            } else {
                constexpr int LR = 64 / RL;                // lanes to a row's chunk
                constexpr int B = FP8 ? 1 : 2;
#pragma unroll
                for (int c = 0; c < NC; ++c)
#pragma unroll
                    for (int i = 0; i < RPG / RL; ++i)
                        wv[t][c * (RPG / RL) + i] = load_nt16(reinterpret_cast<const char*>(w_) + (row_of(i * RL + lane / LR) * K + kw0 + c * 256) * B + (lane % LR) * 16);
                if constexpr (FP8) {
#pragma unroll
                    for (int i = 0; i < 2 * NC; ++i) wsc[t][i] = to_f(a.wscale[(row_of(l15 % RPG) >> 7) * (size_t)(K >> 7) + (kw0 >> 7) + i]);
                }
            }
        }
    };
    const int em = tid >> 4, en = tid & 15;
    float res0 = 0.f;                                      // of the first group; behind the weights, since its address waits for the arguments that are not preloaded
    auto load_res = [&]() {
        if constexpr (EPI == EPI_RESID) res0 = a.res[(size_t)min(em, M - 1) * a.ld_out + min((int)blockIdx.x * RPG + en, N - 1)];
    };

    // ---- activation fragments of this wave's K quarter ----
    // Issue order = arrival order: rows and gamma (L2) are requested BEFORE the weight stream (HBM), so the RMSNorm
    // statistic, its barrier and the bf16 conversion run while the weights are still in flight (the other way round the
    // prologue started when the last weight byte had landed - the batch-1 kernels' lesson).
    uint4 af[S];
    char* img = s_img[wid];
    auto slot = [&](int c8, int m) { return (c8 * MR + (m ^ (c8 & (MR - 1)))) * 16; };
    auto order = []() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); __builtin_amdgcn_wave_barrier(); };
    auto take = [&](int c) {                               // behind the wave's own writes; the next chunk's come behind it
        order();
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const int c8 = FP8 ? 8 * (s >> 1) + 2 * q + (s & 1) : 4 * s + q;
            af[8 * c + s] = *reinterpret_cast<const uint4*>(img + slot(c8, l15 & (MR - 1)));
        }
        order();
    };
    if constexpr (PRO == PRO_NORM) {
        constexpr bool HOLD = MR * NC <= 32;               // raw rows stay in registers across the reduction
        const float* src = x_ + kw0 + 4 * lane;
        auto row = [&](int m, int c) { return *reinterpret_cast<const float4*>(src + (size_t)min(m, M - 1) * K + 256 * c); };
        float4 r[HOLD ? NC : 1][MR];
        uint2 g[NC];
        float ss[MR];
        if constexpr (HOLD) {
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int m = 0; m < MR; ++m) r[c][m] = row(m, c);
        }
#pragma unroll
        for (int c = 0; c < NC; ++c) g[c] = *reinterpret_cast<const uint2*>(gamma_ + kw0 + 256 * c + 4 * lane);
        if constexpr (!HOLD) {
#pragma unroll
            for (int m = 0; m < MR; ++m) ss[m] = 0.f;
            for (int c = 0; c < NC; ++c) {
#pragma unroll
                for (int m = 0; m < MR; ++m) r[0][m] = row(m, c);
#pragma unroll
                for (int m = 0; m < MR; ++m) ss[m] += r[0][m].x * r[0][m].x + r[0][m].y * r[0][m].y + r[0][m].z * r[0][m].z + r[0][m].w * r[0][m].w;
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        load_w(blockIdx.x * RPG);
        load_res();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            if constexpr (HOLD) {
                ss[m] = 0.f;
#pragma unroll
                for (int c = 0; c < NC; ++c) ss[m] += r[c][m].x * r[c][m].x + r[c][m].y * r[c][m].y + r[c][m].z * r[c][m].z + r[c][m].w * r[c][m].w;
            }
        }
        // 16 lanes, 16 (8) rows: at each step a lane keeps the half of the rows that its bit names and hands the other half over, so it ends with row lane & (MR - 1)
        const bool b0 = lane & 1, b1 = lane & 2, b2 = lane & 4, b3 = lane & 8;
        if constexpr (MR == 16) {
#pragma unroll
            for (int i = 0; i < 8; ++i) ss[i] = (b3 ? ss[i + 8] : ss[i]) + dpp_f<DPP_MIRROR>(b3 ? ss[i] : ss[i + 8]);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) ss[i] = (b2 ? ss[i + 4] : ss[i]) + dpp_f<DPP_HALF_MIRROR>(b2 ? ss[i] : ss[i + 4]);
#pragma unroll
        for (int i = 0; i < 2; ++i) ss[i] = (b1 ? ss[i + 2] : ss[i]) + dpp_f<DPP_XOR2>(b1 ? ss[i] : ss[i + 2]);
        ss[0] = (b0 ? ss[1] : ss[0]) + dpp_f<DPP_XOR1>(b0 ? ss[0] : ss[1]);
        if constexpr (MR == 8) ss[0] += dpp_f<DPP_ROR8>(ss[0]);
        const int mr = lane & (MR - 1);                    // a lane's row; the others' come from their lanes
        s_ss[mr][4 * wid + q] = ss[0];
        __syncthreads();
        float tot = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float4 v = *reinterpret_cast<const float4*>(&s_ss[mr][4 * i]);
            tot += (v.x + v.y) + (v.z + v.w);
        }
        const float mine = 1.0f / sqrtf(tot / K + a.eps);
        float inv[MR];
#pragma unroll
        for (int m = 0; m < MR; ++m) inv[m] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(mine), m));
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const float g0 = __uint_as_float(g[c].x << 16), g1 = __uint_as_float(g[c].x & 0xFFFF0000u), g2 = __uint_as_float(g[c].y << 16), g3 = __uint_as_float(g[c].y & 0xFFFF0000u);
            if constexpr (!HOLD) {
#pragma unroll
                for (int m = 0; m < MR; ++m) r[0][m] = row(m, c);
            }
#pragma unroll
            for (int m = 0; m < MR; ++m) {
                const float4 v = r[HOLD ? c : 0][m];
                *reinterpret_cast<uint2*>(img + slot(lane >> 1, m) + (lane & 1) * 8) =
                    make_uint2(pack_bf16x2(v.x * inv[m] * g0, v.y * inv[m] * g1), pack_bf16x2(v.z * inv[m] * g2, v.w * inv[m] * g3));
            }
            take(c);
        }
    } else {                                               // bf16 hand-off: 32 lanes to the 512 bytes of a row's chunk
        const bf16* src = reinterpret_cast<const bf16*>(x_) + kw0 + 8 * (lane & 31);
        u32x4 r[NC][MR / 2];
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int i = 0; i < MR / 2; ++i) r[c][i] = *reinterpret_cast<const u32x4*>(src + (size_t)min(2 * i + (lane >> 5), M - 1) * K + 256 * c);
        __builtin_amdgcn_sched_barrier(0);
        load_w(blockIdx.x * RPG);
        load_res();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < NC; ++c) {
#pragma unroll
            for (int i = 0; i < MR / 2; ++i) *reinterpret_cast<u32x4*>(img + slot(lane & 31, 2 * i + (lane >> 5))) = r[c][i];
            take(c);
        }
    }

    // 8 k of e4m3 codes, scaled
    auto widen = [](uint32_t lo, uint32_t hi, float sc) {
        const f32x2 c0 = __builtin_amdgcn_cvt_pk_f32_fp8((int)lo, false), c1 = __builtin_amdgcn_cvt_pk_f32_fp8((int)lo, true);
        const f32x2 c2 = __builtin_amdgcn_cvt_pk_f32_fp8((int)hi, false), c3 = __builtin_amdgcn_cvt_pk_f32_fp8((int)hi, true);
        return make_uint4(pack_bf16x2(c0.x * sc, c0.y * sc), pack_bf16x2(c1.x * sc, c1.y * sc), pack_bf16x2(c2.x * sc, c2.y * sc), pack_bf16x2(c3.x * sc, c3.y * sc));
    };
    auto half = [&](const uint4& v, int h, float sc) { return h ? widen(v.z, v.w, sc) : widen(v.x, v.y, sc); };
    float bv = -INFINITY;
    int bi = 0x7FFFFFFF;
    for (int g = blockIdx.x; g < ngroups; g += gridDim.x) {
        const int n0 = g * RPG;
        float resv = res0;
        if constexpr (EPI == EPI_RESID) {
            if (g != (int)blockIdx.x) resv = a.res[(size_t)min(em, M - 1) * a.ld_out + min(n0 + en, N - 1)];
        }
        f32x4_b acc[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = f32x4_b{0.f, 0.f, 0.f, 0.f};
        auto mul = [&](int t, int s, const uint4& w) {
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_b, af[s]), __builtin_bit_cast(bf16x8_b, w), acc[t], 0, 0, 0);
        };
        if constexpr (FRAG) {
#pragma unroll
            for (int s = 0; s < S; ++s)
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    if constexpr (FP8) mul(t, s, half(wv[t][s / 2], s & 1, wsc[t][s / 2]));
                    else mul(t, s, wv[t][s]);
                }
        } else {
            constexpr int LR = 64 / RL;
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    auto at = [&](int c16, int r) { return img + (c16 * RPG + (r ^ (c16 & (RPG - 1)))) * 16; };
#pragma unroll
                    for (int i = 0; i < RPG / RL; ++i) *reinterpret_cast<uint4*>(at(lane % LR, i * RL + lane / LR)) = wv[t][c * (RPG / RL) + i];
                    order();
                    uint4 w[FP8 ? 4 : 8];
#pragma unroll
                    for (int s = 0; s < (FP8 ? 4 : 8); ++s) w[s] = *reinterpret_cast<const uint4*>(at(4 * s + q, l15 % RPG));
                    order();
#pragma unroll
                    for (int s = 0; s < 8; ++s) {
                        if constexpr (FP8) mul(t, 8 * c + s, half(w[s / 2], s & 1, wsc[t][2 * c + s / 4]));
                        else mul(t, 8 * c + s, w[s]);
                    }
                }
        }
        // the next group's weights (lm_head: a workgroup walks several groups) travel while this one is reduced and stored
        if (g + (int)gridDim.x < ngroups) load_w((g + (int)gridDim.x) * RPG);
        __syncthreads();                                    // the previous trip's partial tiles have been read
        if (l15 < RPG) {
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) red[((t * 4 + wid) * 16 + q * 4 + r) * 16 + l15] = acc[t][r];
        }
        __syncthreads();
        const bool ok = em < M && en < RPG && n0 + en < N;
        float y[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const float* p = red + (size_t)t * 4 * 256 + em * 16 + en;
            y[t] = ok ? p[0] + p[256] + p[512] + p[768] : 0.f;
        }
        const size_t o = (size_t)em * a.ld_out + n0 + en;
        if constexpr (EPI == EPI_STORE) {
            if (ok) a.out[o] = y[0];
        } else if constexpr (EPI == EPI_RESID) {
            if (ok) a.out[o] = resv + y[0];
        } else if constexpr (EPI == EPI_SWIGLU) {
            if (ok) {
                const float act = y[0] / (1.0f + __expf(-y[0])) * y[NT - 1];
                if (a.out16) a.out16[o] = from_f<bf16>(act);
                else a.out[o] = act;
            }
        } else {   // EPI_LOGITS
            if (ok) {
                a.out[o] = y[0];
                if (y[0] > bv) { bv = y[0]; bi = n0 + en; }
            }
        }
    }
    if constexpr (EPI == EPI_LOGITS) {
#pragma unroll
        for (int off = 8; off >= 1; off >>= 1) {
            const float ov = __shfl_xor(bv, off, 64);
            const int oi = __shfl_xor(bi, off, 64);
            if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
        }
        if (en == 0 && em < M) {
            a.amax_val[(size_t)em * nblk_logits + blockIdx.x] = bv;
            a.amax_idx[(size_t)em * nblk_logits + blockIdx.x] = bi;
        }
    }
    tls.end();
}

// ---------------------------------------------------------------------------------------------------------------------
// M-tiled variant: 17..64 sequences per launch (MT = 2 or 4 tiles of 16 rows), every weight byte still read ONCE.
//
// Chunks of at most 16 sequences made a batch of 64 four full passes over the weights (4 x 1.08 ms per step on
// Qwen3-0.6B).  Here a wave keeps its K quarter of the workgroup's weight rows in registers exactly as above and runs
// MT MFMAs per weight fragment, one per 16-row tile of the batch.  The activation rows arrive as bf16 (the RMSNorm'ed
// rows from norm_rows_bf16, the attention output, the SwiGLU output): an A fragment is one 16-byte load, no conversion,
// no cross-wave reduction before the first MFMA.  S * MT <= 32 fragments stay resident (and are reused by every weight
// group an lm_head workgroup walks); beyond that they stream from L2 in chunks of CH = 4 k-steps, the next chunk's loads
// issued before the current chunk's MFMAs.  Rows >= M of the last tile repeat row M - 1: MFMA output rows are independent
// and the epilogue drops them.

template <class WT, int EPI, int S, int RPG, int MT>
__global__ __launch_bounds__(256) void batched_mt_kernel(unsigned long long* tl, FusedArgs a, int M, int nblk_logits) {
    const TLStamp tls(tl);
    constexpr bool FP8 = std::is_same<WT, fp8e4m3>::value;
    constexpr int NT = (EPI == EPI_SWIGLU) ? 2 : 1;
    constexpr int CH = (S * MT <= 32) ? S : 4;             // k-steps per activation chunk
    constexpr int NCH = S / CH;
    static_assert(S % CH == 0, "chunking");
    __shared__ float red[NT * 4 * MT * 256];               // [NT][4 waves][MT][16 m][16 n]
    const int K = a.K, N = a.N;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, q = lane >> 4, l15 = lane & 15;
    const int ngroups = (N + RPG - 1) / RPG;
    const int kw0 = wid * S * 32;
    const bool wlane = l15 < RPG;
    uint4 wv[NT][S];
    float wsc[NT][S];
    auto load_w = [&](int n0) {
        const int nrow = min(n0 + l15, N - 1);
        if constexpr (!FP8 && RPG == 16) {
            if (a.wp != nullptr && n0 + 16 <= N) {          // fragment-major copy: see batched_reg_kernel
                const int ksn = K >> 5;
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const bf16* run = a.wp + (((size_t)((t == 0 ? n0 : N + n0) >> 4) * ksn + (kw0 >> 5)) * 64 + lane) * 8;
#pragma unroll
                    for (int s = 0; s < S; ++s) wv[t][s] = load_nt16(run + (size_t)s * 512);
                }
                return;
            }
        }
        if (wlane) {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const size_t row = (size_t)(t == 0 ? nrow : N + nrow);
#pragma unroll
                for (int s = 0; s < S; ++s) {
                    const int k = kw0 + s * 32 + 8 * q;
                    if constexpr (FP8) {
                        const uint2 v = *reinterpret_cast<const uint2*>(reinterpret_cast<const uint8_t*>(a.w) + row * K + k);
                        wv[t][s] = make_uint4(v.x, v.y, 0, 0);
                        wsc[t][s] = to_f(a.wscale[(row >> 7) * (size_t)(K >> 7) + (k >> 7)]);
                    } else {
                        wv[t][s] = load_nt16(reinterpret_cast<const bf16*>(a.w) + row * K + k);
                    }
                }
            }
        }
    };
    __builtin_amdgcn_sched_barrier(0);
    load_w(blockIdx.x * RPG);                              // in flight before the activations are touched
    const int em = tid >> 4, en = tid & 15;
    __builtin_amdgcn_sched_barrier(0);

    const bf16* xrow[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) xrow[t] = a.xin16 + (size_t)min(t * 16 + l15, M - 1) * K + kw0 + 8 * q;
    uint4 af[NCH > 1 ? 2 : 1][CH][MT];
    auto load_a = [&](int buf, int c) {
#pragma unroll
        for (int j = 0; j < CH; ++j)
#pragma unroll
            for (int t = 0; t < MT; ++t) af[buf][j][t] = *reinterpret_cast<const uint4*>(xrow[t] + (c * CH + j) * 32);
    };
    if constexpr (NCH == 1) load_a(0, 0);
    auto bfrag = [&](int t, int s) -> uint4 {
        if constexpr (FP8) {
            const f32x2 c0 = __builtin_amdgcn_cvt_pk_f32_fp8((int)wv[t][s].x, false), c1 = __builtin_amdgcn_cvt_pk_f32_fp8((int)wv[t][s].x, true);
            const f32x2 c2 = __builtin_amdgcn_cvt_pk_f32_fp8((int)wv[t][s].y, false), c3 = __builtin_amdgcn_cvt_pk_f32_fp8((int)wv[t][s].y, true);
            const float sc = wsc[t][s];
            return make_uint4(pack_bf16x2(c0.x * sc, c0.y * sc), pack_bf16x2(c1.x * sc, c1.y * sc), pack_bf16x2(c2.x * sc, c2.y * sc),
                              pack_bf16x2(c3.x * sc, c3.y * sc));
        } else {
            return wv[t][s];
        }
    };
    float bv[MT];
    int bi[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) { bv[t] = -INFINITY; bi[t] = 0x7FFFFFFF; }
    for (int g = blockIdx.x; g < ngroups; g += gridDim.x) {
        const int n0 = g * RPG;
        float resv[MT];
        if constexpr (EPI == EPI_RESID) {
#pragma unroll
            for (int t = 0; t < MT; ++t) resv[t] = a.res[(size_t)min(t * 16 + em, M - 1) * a.ld_out + min(n0 + en, N - 1)];
        }
        f32x4_b acc[MT][NT];
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int u = 0; u < NT; ++u) acc[t][u] = f32x4_b{0.f, 0.f, 0.f, 0.f};
        if constexpr (NCH > 1) load_a(0, 0);
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            if constexpr (NCH > 1) { if (c + 1 < NCH) load_a((c + 1) & 1, c + 1); }
#pragma unroll
            for (int j = 0; j < CH; ++j) {
#pragma unroll
                for (int u = 0; u < NT; ++u) {
                    const uint4 b = bfrag(u, c * CH + j);
#pragma unroll
                    for (int t = 0; t < MT; ++t)
                        acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_b, af[c & 1][j][t]),
                                                                             __builtin_bit_cast(bf16x8_b, b), acc[t][u], 0, 0, 0);
                }
            }
        }
        // the next group's weights (lm_head: a workgroup walks several groups) travel while this one is reduced and stored
        if (g + (int)gridDim.x < ngroups) load_w((g + (int)gridDim.x) * RPG);
        __syncthreads();                                    // the previous trip's partial tiles have been read
        if (wlane) {
#pragma unroll
            for (int u = 0; u < NT; ++u)
#pragma unroll
                for (int t = 0; t < MT; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) red[(((u * 4 + wid) * MT + t) * 16 + q * 4 + r) * 16 + l15] = acc[t][u][r];
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            const int m = t * 16 + em;
            const bool ok = m < M && en < RPG && n0 + en < N;
            float y[NT];
#pragma unroll
            for (int u = 0; u < NT; ++u) {
                const float* p = red + ((size_t)(u * 4) * MT + t) * 256 + em * 16 + en;
                y[u] = ok ? (p[0] + p[MT * 256] + p[2 * MT * 256] + p[3 * MT * 256]) : 0.f;
            }
            const size_t o = (size_t)m * a.ld_out + n0 + en;
            if constexpr (EPI == EPI_STORE) {
                if (ok) a.out[o] = y[0];
            } else if constexpr (EPI == EPI_RESID) {
                const float v = resv[t] + y[0];
                if (ok) a.out[o] = v;
            } else if constexpr (EPI == EPI_SWIGLU) {
                if (ok) {
                    const float act = y[0] / (1.0f + __expf(-y[0])) * y[NT - 1];
                    if (a.out16) a.out16[o] = from_f<bf16>(act);
                    else a.out[o] = act;
                }
            } else {   // EPI_LOGITS
                if (ok) {
                    a.out[o] = y[0];
                    if (y[0] > bv[t]) { bv[t] = y[0]; bi[t] = n0 + en; }
                }
            }
        }
    }
    if constexpr (EPI == EPI_LOGITS) {
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            float v = bv[t];
            int ix = bi[t];
#pragma unroll
            for (int off = 8; off >= 1; off >>= 1) {
                const float ov = __shfl_xor(v, off, 64);
                const int oi = __shfl_xor(ix, off, 64);
                if (ov > v || (ov == v && oi < ix)) { v = ov; ix = oi; }
            }
            const int m = t * 16 + em;
            if (en == 0 && m < M) {
                a.amax_val[(size_t)m * nblk_logits + blockIdx.x] = v;
                a.amax_idx[(size_t)m * nblk_logits + blockIdx.x] = ix;
            }
        }
    }
    tls.end();
}

// (Tried for the N = hidden projections at batch 64: 16 rows per workgroup - 64 workgroups, a quarter of the activation
// traffic: 17.2 / 12.1 us against 15.5 / 11.1; and the weights of 16 rows parked in LDS with one wave per 16-row batch tile,
// no cross-wave reduction: 16.4 us average.  A workgroup keeps at most ~64 KB of loads in flight, so 64 workgroups cannot
// pull the 6 MB of weights plus their activation rows faster than 256 four-row workgroups that each re-read the rows.)
static int mt_rows_per_group(int N, int epi) { return (epi == EPI_LOGITS || ceil_div(N, 16) >= 192) ? 16 : 4; }

template <class WT, int EPI, int S>
static pgk_status launch_batched_mt(const FusedArgs& a, int M, hipStream_t st, int nblk_logits) {
    const int rpg = mt_rows_per_group(a.N, EPI);
    const int grid = (EPI == EPI_LOGITS) ? nblk_logits : ceil_div(a.N, rpg);
    const bool two = M <= 32;
    hipError_t he = hipSuccess;
    if constexpr (EPI == EPI_LOGITS) {
        if (two) he = launch_k(batched_mt_kernel<WT, EPI, S, 16, 2>, dim3(grid), dim3(256), 0, st, a, M, nblk_logits);
        else he = launch_k(batched_mt_kernel<WT, EPI, S, 16, 4>, dim3(grid), dim3(256), 0, st, a, M, nblk_logits);
    } else {
        if (rpg == 16 && two) he = launch_k(batched_mt_kernel<WT, EPI, S, 16, 2>, dim3(grid), dim3(256), 0, st, a, M, nblk_logits);
        else if (rpg == 16) he = launch_k(batched_mt_kernel<WT, EPI, S, 16, 4>, dim3(grid), dim3(256), 0, st, a, M, nblk_logits);
        else if (two) he = launch_k(batched_mt_kernel<WT, EPI, S, 4, 2>, dim3(grid), dim3(256), 0, st, a, M, nblk_logits);
        else he = launch_k(batched_mt_kernel<WT, EPI, S, 4, 4>, dim3(grid), dim3(256), 0, st, a, M, nblk_logits);
    }
    PGK_CHECK_HIP(he);
    return PGK_OK;
}

template <class WT, int EPI>
static pgk_status launch_batched_tiled(const FusedArgs& a, int M, hipStream_t st, int nblk_logits = 0) {
    PGK_REQUIRE(a.xin16 != nullptr, "batched decode projection: %d sequences need bf16 input rows", M);
    PGK_REQUIRE(M > 16 && M <= 64, "batched decode projection: tiled kernels take 17..64 sequences, got %d", M);
    switch (a.K / 128) {
        case 2: return launch_batched_mt<WT, EPI, 2>(a, M, st, nblk_logits);
        case 4: return launch_batched_mt<WT, EPI, 4>(a, M, st, nblk_logits);
        case 8: return launch_batched_mt<WT, EPI, 8>(a, M, st, nblk_logits);
        case 16: return launch_batched_mt<WT, EPI, 16>(a, M, st, nblk_logits);
        case 24: return launch_batched_mt<WT, EPI, 24>(a, M, st, nblk_logits);
        case 32: return launch_batched_mt<WT, EPI, 32>(a, M, st, nblk_logits);
    }
    return set_error(PGK_ERR_UNSUPPORTED, "batched decode projection: K=%d is not 128 x {2,4,8,16,24,32}", a.K);
}

template <class WT, int PRO, int EPI, int S, int RPG>
static pgk_status launch_batched_rows(const FusedArgs& a, int M, int grid, hipStream_t st, int nblk_logits) {
    const float* x = PRO == PRO_NORM ? a.h : reinterpret_cast<const float*>(a.xin16);
    hipError_t he;
    if (M <= 8) he = launch_k(batched_reg_kernel<WT, PRO, EPI, S, RPG, 8>, dim3(grid), dim3(256), 0, st, a.w, a.wp, x, a.gamma, a.N, a.K, M, nblk_logits, a);
    else he = launch_k(batched_reg_kernel<WT, PRO, EPI, S, RPG, 16>, dim3(grid), dim3(256), 0, st, a.w, a.wp, x, a.gamma, a.N, a.K, M, nblk_logits, a);
    PGK_CHECK_HIP(he);
    return PGK_OK;
}

template <class WT, int PRO, int EPI, int S>
static pgk_status launch_batched_reg(const FusedArgs& a, int M, hipStream_t st, int nblk_logits) {
    // enough workgroups to pull HBM bandwidth: fewer weight rows per workgroup when N / 16 would leave CUs idle
    const int rpg = (EPI == EPI_LOGITS || ceil_div(a.N, 16) >= 192) ? 16 : (ceil_div(a.N, 8) >= 192 ? 8 : 4);
    if constexpr (EPI == EPI_LOGITS) return launch_batched_rows<WT, PRO, EPI, S, 16>(a, M, nblk_logits, st, nblk_logits);
    else {
        const int grid = ceil_div(a.N, rpg);
        if (rpg == 16) return launch_batched_rows<WT, PRO, EPI, S, 16>(a, M, grid, st, nblk_logits);
        if (rpg == 8) return launch_batched_rows<WT, PRO, EPI, S, 8>(a, M, grid, st, nblk_logits);
        return launch_batched_rows<WT, PRO, EPI, S, 4>(a, M, grid, st, nblk_logits);
    }
}

template <class WT, int PRO, int EPI, int MP>
static pgk_status launch_batched_image(const FusedArgs& a, int M, int steps, int grid, size_t lds, hipStream_t st, int nblk_logits) {
    static bool done = false;
    if (lds > 48 * 1024 && !done) {
        PGK_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&batched_mfma_kernel<WT, PRO, EPI, MP>),
                                          hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024 - 2048));
        done = true;
    }
    PGK_CHECK_HIP(launch_k(batched_mfma_kernel<WT, PRO, EPI, MP>, dim3(grid), dim3(256), lds, st, a, M, steps, nblk_logits));
    return PGK_OK;
}

template <class WT, int PRO, int EPI>
static pgk_status launch_batched(const FusedArgs& a, int M, hipStream_t st, int nblk_logits = 0) {
    PGK_REQUIRE(a.K % 128 == 0 && M >= 1 && M <= 16, "batched decode projection: K=%d must be a multiple of 128 and M=%d in [1,16]", a.K, M);
    PGK_REQUIRE(PRO == PRO_NORM ? a.h != nullptr : a.xin16 != nullptr, "batched decode projection: no input rows");
    const int steps = a.K / 128, ngroups = ceil_div(a.N, 16);
    // register-resident activations at the instantiated widths; the LDS-image kernel below for every other K
    if (steps == 8) return launch_batched_reg<WT, PRO, EPI, 8>(a, M, st, nblk_logits);
    if (steps == 16) return launch_batched_reg<WT, PRO, EPI, 16>(a, M, st, nblk_logits);
    if (steps == 24) return launch_batched_reg<WT, PRO, EPI, 24>(a, M, st, nblk_logits);
    if (steps == 32) return launch_batched_reg<WT, PRO, EPI, 32>(a, M, st, nblk_logits);
    // the prologue (RMSNorm of the M rows) is per workgroup: large N (lm_head) runs 2048 workgroups over several groups each
    const int grid = (EPI == EPI_LOGITS) ? nblk_logits : ngroups;
    constexpr int NT = (EPI == EPI_SWIGLU) ? 2 : 1;
    const int mp = M <= 8 ? 8 : 16;
    const size_t lds = (size_t)(a.K / 8) * mp * 16 + (size_t)NT * 4 * 256 * 4;
    PGK_REQUIRE(lds <= 158 * 1024, "batched decode projection: K=%d does not fit the LDS image", a.K);
    if (mp == 8) return launch_batched_image<WT, PRO, EPI, 8>(a, M, steps, grid, lds, st, nblk_logits);
    return launch_batched_image<WT, PRO, EPI, 16>(a, M, steps, grid, lds, st, nblk_logits);
}
