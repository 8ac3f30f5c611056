// Decode projections of wide models on the matrix pipe: 1..8 sequences, every weight byte read once.
//
// Bound by HBM: gate/up of a 4096-wide layer is 235 MB (bf16) or 117 MB (e4m3).  The GEMV kernels of engine.hip stream a long row at 6 TB/s
// once they stream, but their any-K prologue ran 15-20 us in front of that (element loads, a serial sum over 8 o_proj partial vectors in
// each of 1024 workgroups), and they take 1, 2 or 4 sequences: six took two passes over the weights.  Here
//   * one workgroup of 8 waves per CU owns N / 256 output rows; the waves split K eight ways, so that each holds its slice of the
//     activations as matrix operands in registers for all of the workgroup's rows;
//   * a wave's weight loads are 4 rows x 256 contiguous bytes, 16 KiB in flight per wave (128 KiB per CU: 5 us of its share of HBM), issued
//     before the activations are touched; a 16-row chunk passes through 4 KiB of the wave's own LDS (swizzled, no barrier) into the operand
//     layout of v_mfma_f32_16x16x32_bf16.  Loading that layout directly would be 16 pieces of 64 bytes per instruction, which a CU's
//     texture path takes three times as long for;
//   * fp32 activations are split into three bf16 pieces each (24 bits, as the fp32 products they replace), which take rows of the 16-row operand
//     that few sequences leave free: all three for up to four sequences; for up to eight the first two, and the third are a second operand for
//     the same weights (the matrix pipe has the time); e4m3 weights are exact in bf16 and their block scales multiply fp32 sums;
//   * 1 / rms is a factor of the finished sums, so no wave waits for the row statistic.
//
// Measured on the Llama-3-8B shape, us per launch (before: the GEMV kernels; bf16 with 6 sequences took two launches, of 4 and of 2):
//                 bytes (bf16)   bf16, 1 sequence   bf16, 6 sequences   e4m3, 1 sequence
//     qkv              50 MB       19.4 -> 11.1         65.2 -> 12.3       19.1 ->  8.6
//     o_proj           34 MB       (merged)  8.3        (merged)  8.9      (merged) 5.8   (7.5 with the merge of split attention's records, a launch of 5 before)
//     gate/up         235 MB       82.7 -> 37.5        193.4 -> 38.1       67.2 -> 23.3
//     down            117 MB       37.9 -> 20.0        107.9 -> 27.2       39.5 -> 12.9
//     lm_head        1051 MB      171.2 -> 162.8       371.0 -> 169        (bf16)
// (5..7 sequences: with two pieces, 16 bits, 12, 8.6, 37.7, 24.6 and 169; the pieces of down's input, read by every workgroup, are what six cost more
// than one.)
// i.e. 6.2 TB/s on gate/up and 6.4 on lm_head.  One step: 5.34 -> 3.05 ms, 15.3 -> 3.43 ms, 4.68 -> 2.04 ms (context 700, 1100, 700).

#include <algorithm>

#include "wide.hip.h"

namespace pgk {

namespace {

constexpr int WD_WAVES = 8, WD_THREADS = WD_WAVES * 64;
constexpr int WD_TILES = 7;                      // 16-row tiles between two reductions over the waves (4 KiB of LDS each)
constexpr int WD_RED = WD_WAVES * 8 * 16;        // floats of one tile: [wave][8 sequences][16 rows]

typedef __bf16 bf16x8_w __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_w __attribute__((ext_vector_type(2)));
typedef float f32x4_w __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(4))) uint32_t* scalar_u32;

struct WideArgs {
    float eps;
    float* out;
    int ld_out;
    const bf16* pieces_in;
    bf16* pieces_out;
    float* amax_val;
    int* amax_idx;
    const float* part;       // WIDE_NORM_SUM: [parts][K]; WIDE_MERGE: [K / ld_out heads][parts][2 + ld_out]
    int parts;
    float* h_out;
};

__device__ __forceinline__ f32x4_w mfma_w(const uint4& a, const uint4& b, f32x4_w c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_w, a), __builtin_bit_cast(bf16x8_w, b), c, 0, 0, 0);
}
__device__ __forceinline__ uint32_t widen2(uint32_t codes, bool hi) {
    const bf16x2_w r = hi ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((int)codes, 1.0f, true) : __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((int)codes, 1.0f, false);
    return __builtin_bit_cast(uint32_t, r);
}
__device__ __forceinline__ uint4 widen8(uint32_t lo, uint32_t hi) { return make_uint4(widen2(lo, false), widen2(lo, true), widen2(hi, false), widen2(hi, true)); }
// The pieces of a value are its leading bits, cut off: three hold all 24 of them, and a value beyond the largest bf16 does not become an
// infinity.  What the first piece leaves of a value (an infinity is one piece; what the others leave is a plain difference):
__device__ __forceinline__ float rest(float v, float piece) { const float d = v - piece; return d == d ? d : 0.f; }
__device__ __forceinline__ uint32_t cut2(float lo, float hi) { return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u); }
// LDS of one wave: its lanes write and read in program order, the compiler must keep that order
__device__ __forceinline__ void wave_order() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); __builtin_amdgcn_wave_barrier(); }

// LDS bytes of a wave: 16 operand rows of `rs` bytes on their way to registers, afterwards two chunks of weights and, with eight sequence slots, the
// third pieces of a row each (rs = 0: the operands come from memory)
constexpr int wide_scratch(int rs, int mt) {
    const int rows = 16 * rs, body = 8192 + (mt == 8 ? 8 * rs : 0);
    return rows > body ? rows : body;
}

// where element k of a row lies among the pieces: 32-k block, quarter, position (e4m3: a lane's 16 codes are two steps of 8)
template <bool FP8> __device__ __forceinline__ void piece_of(int k, int& blk, int& q, int& j) {
    if constexpr (FP8) { blk = (k >> 6) * 2 + ((k >> 3) & 1); q = (k >> 4) & 3; }
    else { blk = k >> 5; q = (k >> 3) & 3; }
    j = k & 7;
}

// CH: chunks of 256 weight bytes per row and wave (0: run time, WIDE_PIECES only); MT: sequence slots; NP: WIDE_NORM_SUM's partial vectors, WIDE_MERGE's slices, requested at once.
// rows: output rows (SWIGLU: pairs) of a workgroup, a multiple of 8.
template <class WT, int SRC, int EPI, int CH, int MT, int NP = 1>
__global__ __launch_bounds__(WD_THREADS) void wide_kernel(unsigned long long* tl, const void* w_, const bf16* wscale_, const float* x_, const bf16* gamma_, int N, int rows, int M,
                                                          int K, WideArgs a) {
    const TLStamp tls(tl);
    constexpr bool FP8 = std::is_same<WT, fp8e4m3>::value, REG = SRC != WIDE_PIECES, SUM = SRC == WIDE_NORM_SUM, MERGE = SRC == WIDE_MERGE, NORM = SRC == WIDE_NORM || SUM;
    static_assert(MT == 1 || !(SUM || MERGE), "partial vectors and records of one sequence");
    constexpr int KCH = 256 / sizeof(WT), STEPS = KCH / 32;      // k and matrix steps of a chunk
    constexpr int NS = 3, SS = MT < 8 ? 4 : 8;                   // pieces; operand rows s * SS + m
    // The third pieces of eight rows are an operand of their own: rows m those of an even step, rows 8 + m those of the step after it, and only
    // the products with the weights of the same step count
    constexpr bool TWO = MT == 8;
    constexpr int RD = REG || !FP8 ? 4 : 2;                              // chunks in flight per wave
    constexpr int SL = REG ? CH * KCH : 0, RS = SL * 2 + 16;     // k slice of a wave; LDS row of its pieces (16 bytes on: rows start in different banks)
    constexpr int SCRATCH = wide_scratch(REG ? RS : 0, MT);
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), q = lane >> 4, n16 = lane & 15;
    char* scratch = smem + wid * SCRATCH;
    float* red = reinterpret_cast<float*>(smem + WD_WAVES * SCRATCH);
    __shared__ float s_ss[WD_WAVES][8];
    const int r0 = blockIdx.x * rows, nr = min(rows, N - r0);
    constexpr int PER = EPI == EPI_SWIGLU ? 8 : 16;              // outputs of a tile
    const int T = (nr + PER - 1) / PER;
    const int kb = MERGE ? (int)blockIdx.y * WIDE_RUN : 0, KL = MERGE ? min(WIDE_RUN, K - kb) : K;      // this workgroup's columns
    const int nch = KL / KCH;
    constexpr int CHW = CH > 0 ? CH : 1;
    const int cw = REG ? CH : (nch + WD_WAVES - 1) / WD_WAVES;
    const int c0 = wid * cw;
    const int ncw = REG ? CH : max(0, min(cw, nch - c0));        // chunks of this wave (REG: chunks beyond K multiply zeros)
    const int total = T * ncw;
    constexpr bool GROUPS = EPI == EPI_LOGITS;                   // more than WD_TILES tiles: reduced in groups

    // ---- the activations' loads first: they come from L2 and return before the weights ----
    constexpr int XI = REG ? SL / 256 : 1;
    float4 xv[REG ? MT : 1][XI];
    uint2 gv[XI];
    if constexpr (REG && !MERGE) {
#pragma unroll
        for (int i = 0; i < XI; ++i) {
            const int k = min(c0 * KCH + i * 256 + lane * 4, K - 4);
            if constexpr (NORM) gv[i] = *reinterpret_cast<const uint2*>(gamma_ + k);
#pragma unroll
            for (int m = 0; m < MT; ++m) xv[m][i] = *reinterpret_cast<const float4*>(x_ + (size_t)min(m, M - 1) * K + k);
        }
    }
    float4 pv[SUM || MERGE ? NP : 1][XI];
    if constexpr (SUM) {
#pragma unroll
        for (int p = 0; p < NP; ++p)
#pragma unroll
            for (int i = 0; i < XI; ++i) pv[p][i] = *reinterpret_cast<const float4*>(a.part + (size_t)min(p, a.parts - 1) * K + min(c0 * KCH + i * 256 + lane * 4, K - 4));
    }
    // Records of the wave's heads: values four to a lane, (m, l) of slice `lane` to a lane
    constexpr int HPW = MERGE ? 4 : 1;                           // 64-column quarters of the slice; D = 128: of two heads
    float2 ml[HPW];
    struct __attribute__((packed, aligned(8))) Four { float v[4]; };      // (a record's values start 8 bytes off a 16-byte line)
    if constexpr (MERGE) {
        static_assert(!MERGE || XI == 1, "a wave's slice is 256 columns");
        const int D = a.ld_out, rs = D + 2, k = min(kb + c0 * KCH + lane * 4, K - 4), first = min(kb + c0 * KCH, K - 256);
#pragma unroll
        for (int h = 0; h < HPW; ++h) ml[h] = *reinterpret_cast<const float2*>(a.part + ((size_t)((first + 64 * h) / D) * a.parts + min(lane, a.parts - 1)) * rs);
        const float* rec = a.part + (size_t)(k / D) * a.parts * rs + 2 + k % D;
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const Four f = *reinterpret_cast<const Four*>(rec + (size_t)min(p, a.parts - 1) * rs);
            pv[p][0] = make_float4(f.v[0], f.v[1], f.v[2], f.v[3]);
        }
    }
    const int en = threadIdx.x & (PER - 1), em = (threadIdx.x / PER) & 7, et = threadIdx.x / (PER * 8);
    constexpr int ET = WD_THREADS / (PER * 8);                   // tiles an epilogue trip covers
    float resv = 0.f;
    if constexpr (EPI == EPI_RESID) resv = a.out[(size_t)min(em, M - 1) * a.ld_out + min(r0 + et * 16 + en, N - 1)];

    // ---- weight loads ----
    uint4 rb[RD][4];
    uint4 ra[REG ? 1 : RD][REG ? 1 : STEPS], rc[REG || !TWO ? 1 : RD][REG || !TWO ? 1 : STEPS / 2];  // first pieces, third ones
    uint32_t sc0[FP8 ? RD : 1], sc1[FP8 ? RD : 1];
    const int am = (n16 & (SS - 1)) < MT ? (n16 & (SS - 1)) : 0, as = (n16 / SS) < NS ? n16 / SS : 0;   // this lane's operand row: sequence slot, piece
    // Rows come in groups of 8 (N and `rows` are multiples of 8): a half tile beyond the workgroup's rows reads the other half again.
    // Addresses are a wave-uniform base plus one offset per lane.
    auto half_row = [&](int t, int h) -> int {
        if constexpr (EPI == EPI_SWIGLU) return h * N + r0 + t * 8;
        else return r0 + t * 16 + (t * 16 + 8 * h < nr ? 8 * h : 0);
    };
    const uint32_t w_lane = (uint32_t)q * K * sizeof(WT) + n16 * 16;
    const int pm = min(am, M - 1), p_step = M * NS * 64;         // (slots without a sequence read the last one's pieces again)
    const uint32_t p_lane = (((pm * NS + as) * 4 + q) * 8) * 2, p_third = (((pm * NS + 2) * 4 + q) * 8) * 2 + (n16 >> 3) * p_step;
    int lt = 0, lj = 0;                                          // tile and chunk of the next load
    auto issue_weights = [&](int u) {
        const int ch = REG ? min(c0 + lj, nch - 1) : c0 + lj;
        const int row[2] = {half_row(lt, 0), half_row(lt, 1)};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const char* base = reinterpret_cast<const char*>(w_) + ((size_t)(row[i >> 1] + (i & 1) * 4) * K * sizeof(WT) + (size_t)kb * sizeof(WT) + (size_t)ch * 256);
            rb[u][i] = load_nt16(base + w_lane);
        }
        if constexpr (FP8) {                                     // both scales of the chunk in one word; the halves of a tile may lie in different blocks
            sc0[u] = *(scalar_u32)(wscale_ + (size_t)(row[0] >> 7) * (K >> 7) + (kb >> 7) + ch * 2);
            sc1[u] = *(scalar_u32)(wscale_ + (size_t)(row[1] >> 7) * (K >> 7) + (kb >> 7) + ch * 2);
        }
        if constexpr (REG) { if (++lj == ncw) { lj = 0; ++lt; } }
    };
    auto issue_pieces = [&](int u) {
        if constexpr (!REG) {
            const char* base = reinterpret_cast<const char*>(a.pieces_in) + (size_t)(c0 + lj) * STEPS * p_step;
#pragma unroll
            for (int s = 0; s < STEPS; ++s) ra[u][s] = *reinterpret_cast<const uint4*>(base + s * p_step + p_lane);
            if constexpr (TWO) {
#pragma unroll
                for (int s = 0; s < STEPS; s += 2) rc[u][s / 2] = *reinterpret_cast<const uint4*>(base + s * p_step + p_third);
            }
            if (++lj == ncw) { lj = 0; ++lt; }
        }
    };
#pragma unroll
    for (int u = 0; u < RD; ++u)
        if (u < total) { issue_weights(u); issue_pieces(u); }
    __builtin_amdgcn_sched_barrier(0);

    // ---- activations -> pieces -> operands in registers ----
    uint4 A[REG ? CH * STEPS : 1];
    char* third = scratch + 8192;                                // [8 sequences][RS], behind the weights' chunks
    if constexpr (SUM) {
#pragma unroll
        for (int p = 0; p < NP; ++p)
            if (p < a.parts) {
#pragma unroll
                for (int i = 0; i < XI; ++i) { xv[0][i].x += pv[p][i].x; xv[0][i].y += pv[p][i].y; xv[0][i].z += pv[p][i].z; xv[0][i].w += pv[p][i].w; }
            }
        if (blockIdx.x == 0) {
#pragma unroll
            for (int i = 0; i < XI; ++i)
                if (const int k = c0 * KCH + i * 256 + lane * 4; k < K) *reinterpret_cast<float4*>(a.h_out + k) = xv[0][i];
        }
    }
    if constexpr (MERGE) {                                       // the arithmetic of attn_merge_kernel, slice after slice
        float w[HPW], inv[HPW];
#pragma unroll
        for (int h = 0; h < HPW; ++h) {
            const float m = lane < a.parts ? ml[h].x : -INFINITY, l = lane < a.parts ? ml[h].y : 0.f, mx = wave_max(m);
            w[h] = m == -INFINITY ? 0.f : __expf(m - mx);
            const float tot = wave_sum(w[h] * l);
            inv[h] = tot > 0.f ? 1.0f / tot : 0.f;
        }
        float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
        const int h = lane >> 4;                                 // 64 columns are 16 lanes
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            float ws = 0.f;
#pragma unroll
            for (int x = 0; x < HPW; ++x) {
                const float wx = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w[x]), p));
                ws = h == x ? wx : ws;
            }
            if (p < a.parts) { o.x = fmaf(ws, pv[p][0].x, o.x); o.y = fmaf(ws, pv[p][0].y, o.y); o.z = fmaf(ws, pv[p][0].z, o.z); o.w = fmaf(ws, pv[p][0].w, o.w); }
        }
        float one = inv[0];
#pragma unroll
        for (int x = 1; x < HPW; ++x) one = h == x ? inv[x] : one;
        xv[0][0] = make_float4(o.x * one, o.y * one, o.z * one, o.w * one);
    }
    if constexpr (REG) {
        uint2 p3[TWO ? MT : 1][XI];
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            if (MT > 1 && m >= M) break;                         // (uniform) rows nobody reads the sums of
            float ss = 0.f;
#pragma unroll
            for (int i = 0; i < XI; ++i) {
                float v[4] = {xv[m][i].x, xv[m][i].y, xv[m][i].z, xv[m][i].w};
                if (c0 * KCH + i * 256 + lane * 4 >= KL) v[0] = v[1] = v[2] = v[3] = 0.f;
                if constexpr (NORM) {
                    const float g[4] = {__uint_as_float(gv[i].x << 16), __uint_as_float(gv[i].x & 0xFFFF0000u), __uint_as_float(gv[i].y << 16), __uint_as_float(gv[i].y & 0xFFFF0000u)};
#pragma unroll
                    for (int e = 0; e < 4; ++e) { ss = fmaf(v[e], v[e], ss); v[e] *= g[e]; }
                }
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    const uint32_t p0 = cut2(v[0], v[1]), p1 = cut2(v[2], v[3]);
                    if (TWO && s == 2) { p3[TWO ? m : 0][i] = make_uint2(p0, p1); continue; }
                    *reinterpret_cast<uint2*>(scratch + (s * SS + m) * RS + (i * 256 + lane * 4) * 2) = make_uint2(p0, p1);
                    const float p[4] = {__uint_as_float(p0 << 16), __uint_as_float(p0 & 0xFFFF0000u), __uint_as_float(p1 << 16), __uint_as_float(p1 & 0xFFFF0000u)};
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = s == 0 ? rest(v[e], p[e]) : v[e] - p[e];
                }
            }
            if constexpr (NORM) {
                ss = wave_sum(ss);
                if (lane == 0) s_ss[wid][m] = ss;
            }
        }
        wave_order();
        const char* mine = scratch + (as * SS + am) * RS;
#pragma unroll
        for (int j = 0; j < CH; ++j)
#pragma unroll
            for (int s = 0; s < STEPS; ++s) {
                const int k = FP8 ? j * KCH + (s >> 1) * 64 + q * 16 + (s & 1) * 8 : j * KCH + s * 32 + q * 8;
                A[j * STEPS + s] = *reinterpret_cast<const uint4*>(mine + k * 2);
            }
        wave_order();
        if constexpr (TWO) {
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int i = 0; i < XI; ++i) if (m < M) *reinterpret_cast<uint2*>(third + m * RS + (i * 256 + lane * 4) * 2) = p3[m][i];
        }
    }
    const char* third_row = third + (REG && TWO ? am * RS + (FP8 ? q * 16 + (n16 >> 3) * 8 : (n16 >> 3) * 32 + q * 8) * 2 : 0);

    // ---- body ----
    f32x4_w acc = {0.f, 0.f, 0.f, 0.f}, acc3[2] = {acc, acc};             // acc3: TWO's products, even and odd steps
    int ct = 0, cj = 0, base_t = 0;                              // tile and chunk being multiplied; first tile of the reduction group
    float best_v = -INFINITY;
    int best_i = 0x7FFFFFFF;
    auto put_tile = [&]() {                                      // sum the pieces' rows, leave [sequence][row] for the reduction
        float* dst = red + (size_t)(ct - base_t) * WD_RED + wid * 128;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float v = acc[r];
            if constexpr (MT < 8) { v = q < 3 ? v : 0.f; v += __shfl_xor(v, 16, 64); }
            if constexpr (TWO) v += q < 2 ? acc3[0][r] : acc3[1][r];
            v += __shfl_xor(v, 32, 64);
            if (MT < 8 ? (q == 0 && r < MT) : q < 2) dst[((MT < 8 ? 0 : q * 4) + r) * 16 + n16] = v;
        }
        acc = acc3[0] = acc3[1] = f32x4_w{0.f, 0.f, 0.f, 0.f};
    };
    auto reduce = [&](int nt) {                                  // tiles [base_t, base_t + nt): sum the waves, epilogue
        __syncthreads();
        float inv = 1.f;
        if constexpr (NORM) {
            float t = 0.f;
#pragma unroll
            for (int w = 0; w < WD_WAVES; ++w) t += s_ss[w][em < MT ? em : 0];
            inv = 1.0f / sqrtf(t / K + a.eps);
        }
        for (int tt = et; tt < nt; tt += ET) {
            const float* src = red + (size_t)tt * WD_RED + em * 16 + en;
            float y = 0.f, y2 = 0.f;
#pragma unroll
            for (int w = 0; w < WD_WAVES; ++w) { y += src[w * 128]; if constexpr (EPI == EPI_SWIGLU) y2 += src[w * 128 + 8]; }
            y *= inv;
            const int n = r0 + (base_t + tt) * PER + en;
            if (em < M && n < N && n < r0 + nr) {
                if constexpr (EPI == EPI_SWIGLU) {
                    float v = y / (1.0f + __expf(-y)) * (y2 * inv);
                    int blk, pq, pj;
                    piece_of<FP8>(n, blk, pq, pj);
                    bf16* dst = a.pieces_out + ((((size_t)blk * M + em) * NS) * 4 + pq) * 8 + pj;
#pragma unroll
                    for (int s = 0; s < NS; ++s) {
                        const uint16_t p = (uint16_t)(__float_as_uint(v) >> 16);
                        dst[s * 32] = bf16{p};
                        v = s == 0 ? rest(v, bf16_bits_to_f(p)) : v - bf16_bits_to_f(p);
                    }
                } else if constexpr (EPI == EPI_RESID) {
                    float* o = a.out + (size_t)em * a.ld_out + n;
                    *o = (base_t + tt == et ? resv : *o) + y;
                } else {
                    a.out[MERGE ? (size_t)blockIdx.y * N + n : (size_t)em * a.ld_out + n] = y;
                    if constexpr (EPI == EPI_LOGITS) { if (y > best_v) { best_v = y; best_i = n; } }
                }
            }
        }
        base_t += nt;
    };
    auto step = [&](int u, int opnd, bool more) {                // multiply the chunk in rb[u]; `more`: request the one RD items on
        char* s4 = scratch + (u & 1) * 4096;
#pragma unroll
        for (int i = 0; i < 4; ++i) *reinterpret_cast<uint4*>(s4 + (i * 4 + q) * 256 + ((n16 ^ (i * 4 + q)) * 16)) = rb[u][i];
        auto af = [&](int s) -> const uint4& { return REG ? A[REG ? opnd * STEPS + s : 0] : ra[REG ? 0 : u][REG ? 0 : s]; };
        auto cf = [&](int s) -> uint4 {                          // third pieces of steps s and s + 1
            if constexpr (!REG) return rc[TWO ? u : 0][TWO ? s / 2 : 0];
            else return *reinterpret_cast<const uint4*>(third_row + (opnd * KCH + s * 32) * 2);
        };
        uint32_t w0 = 0, w1 = 0;
        if constexpr (FP8) { w0 = sc0[u]; w1 = sc1[u]; }
        if (more) issue_weights(u);
        wave_order();
        uint4 f[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) f[b] = *reinterpret_cast<const uint4*>(s4 + n16 * 256 + (((b * 4 + q) ^ n16) * 16));
        wave_order();
        if constexpr (FP8) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {                        // a 128-k scale block
                f32x4_w p = {0.f, 0.f, 0.f, 0.f}, p3[2] = {p, p};
#pragma unroll
                for (int b = 2 * h; b < 2 * h + 2; ++b) {
                    const uint4 lo = widen8(f[b].x, f[b].y), hi = widen8(f[b].z, f[b].w);
                    p = mfma_w(af(2 * b), lo, p);
                    p = mfma_w(af(2 * b + 1), hi, p);
                    if constexpr (TWO) {
                        const uint4 c = cf(2 * b);
                        p3[0] = mfma_w(c, lo, p3[0]);
                        p3[1] = mfma_w(c, hi, p3[1]);
                    }
                }
                const uint32_t w = n16 < 8 ? w0 : w1;
                const float sc = h ? __uint_as_float(w & 0xFFFF0000u) : __uint_as_float(w << 16);
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[r] = fmaf(sc, p[r], acc[r]);
                if constexpr (TWO) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) { acc3[0][r] = fmaf(sc, p3[0][r], acc3[0][r]); acc3[1][r] = fmaf(sc, p3[1][r], acc3[1][r]); }
                }
            }
        } else {
#pragma unroll
            for (int b = 0; b < 4; b += 2) {
                acc = mfma_w(af(b), f[b], acc);
                acc = mfma_w(af(b + 1), f[b + 1], acc);
                if constexpr (TWO) {
                    const uint4 c = cf(b);
                    acc3[0] = mfma_w(c, f[b], acc3[0]);
                    acc3[1] = mfma_w(c, f[b + 1], acc3[1]);
                }
            }
        }
        if (more) issue_pieces(u);
        __builtin_amdgcn_sched_barrier(0);                       // keep the next chunk's LDS traffic out of this one: registers
        if (REG ? opnd == CHW - 1 : ++cj == ncw) {
            put_tile();
            cj = 0; ++ct;
            if constexpr (GROUPS) { if (ct - base_t == WD_TILES && ct < T) { reduce(WD_TILES); __syncthreads(); } }
        }
    };
    int base = 0;
    for (; base + 2 * RD <= total; base += RD)
#pragma unroll
        for (int u = 0; u < RD; ++u) step(u, u % CHW, true);
    for (; base < total; base += RD)
#pragma unroll
        for (int u = 0; u < RD; ++u)
            if (base + u < total) step(u, u % CHW, base + u + RD < total);
    if (!REG && ncw == 0)                                        // a wave without a slice adds zeros
        for (; ct < T; ++ct) put_tile();
    reduce(T - base_t);
    if constexpr (EPI == EPI_LOGITS) {
        float* sv = red;
        int* si = reinterpret_cast<int*>(red + WD_THREADS);
        __syncthreads();
        sv[threadIdx.x] = best_v; si[threadIdx.x] = best_i;
        __syncthreads();
        if (threadIdx.x < M) {
            float bv = -INFINITY;
            int bi = 0x7FFFFFFF;
            for (int i = 0; i < ET * 16; ++i) {
                const int at = (i >> 4) * 128 + threadIdx.x * 16 + (i & 15);
                if (sv[at] > bv || (sv[at] == bv && si[at] < bi)) { bv = sv[at]; bi = si[at]; }
            }
            a.amax_val[(size_t)threadIdx.x * gridDim.x + blockIdx.x] = bv;
            a.amax_idx[(size_t)threadIdx.x * gridDim.x + blockIdx.x] = bi;
        }
    }
    tls.end();
}

template <class WT, int SRC, int EPI, int CH, int MT, int NP = 1>
pgk_status launch_wide(const FusedArgs& a, bf16* pieces, int M, int cu_count, int* n_blk, hipStream_t st) {
    constexpr int KCH = 256 / sizeof(WT);
    constexpr int RS = CH * KCH * 2 + 16;
    constexpr int SCRATCH = wide_scratch(SRC != WIDE_PIECES ? RS : 0, MT);
    constexpr int LDS = WD_WAVES * SCRATCH + WD_TILES * WD_RED * 4;
    static_assert(LDS + 512 <= 160 * 1024, "wide_kernel: LDS");
    auto kfn = &wide_kernel<WT, SRC, EPI, CH, MT, NP>;
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kfn), hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
    PGK_CHECK_HIP(attr);
    // one workgroup per CU while its tiles fit one reduction; the vocabulary is reduced in groups
    const int runs = SRC == WIDE_MERGE ? wide_merge_parts(a.K) : 1;
    int rows = wide_rows(a.N, cu_count, runs);
    constexpr int MOST = WD_TILES * (EPI == EPI_SWIGLU ? 8 : 16);
    if (EPI != EPI_LOGITS && rows > MOST) rows = ceil_div(ceil_div(a.N, ceil_div(rows, MOST) * cu_count), 8) * 8;
    const int grid = ceil_div(a.N, rows);
    if (n_blk) *n_blk = grid;
    WideArgs wa{a.eps, a.out, a.ld_out, pieces, pieces, a.amax_val, a.amax_idx, a.part, a.nsplit, a.h_out};
    PGK_CHECK_HIP(launch_k(kfn, dim3(grid, runs), dim3(WD_THREADS), LDS, st, a.w, a.wscale, SRC == WIDE_NORM || SRC == WIDE_NORM_SUM ? a.h : a.xin, a.gamma, a.N, rows, M, a.K, wa));
    return PGK_OK;
}

template <class WT, int SRC, int EPI, int CH>
pgk_status launch_wide_m(const FusedArgs& a, bf16* pieces, int M, int cu_count, int* n_blk, hipStream_t st) {
    if (M == 1) return launch_wide<WT, SRC, EPI, CH, 1>(a, pieces, M, cu_count, n_blk, st);
    if (M <= 4) return launch_wide<WT, SRC, EPI, CH, 4>(a, pieces, M, cu_count, n_blk, st);
    return launch_wide<WT, SRC, EPI, CH, 8>(a, pieces, M, cu_count, n_blk, st);
}

template <class WT, int SRC, int EPI>
pgk_status launch_wide_k(const FusedArgs& a, bf16* pieces, int M, int cu_count, int* n_blk, hipStream_t st) {
    if constexpr (SRC == WIDE_PIECES) return launch_wide_m<WT, SRC, EPI, 0>(a, pieces, M, cu_count, n_blk, st);
    else {
        constexpr int F = std::is_same<WT, fp8e4m3>::value ? 2 : 1;      // a slice of 256 or 512 k per wave
        if (a.K <= 2048) return launch_wide_m<WT, SRC, EPI, 2 / F>(a, pieces, M, cu_count, n_blk, st);
        return launch_wide_m<WT, SRC, EPI, 4 / F>(a, pieces, M, cu_count, n_blk, st);
    }
}

template <class WT>
pgk_status launch_wide_e(int src, int epi, const FusedArgs& a, bf16* pieces, int M, int cu_count, int* n_blk, hipStream_t st) {
    if (src == WIDE_NORM && epi == EPI_STORE) return launch_wide_k<WT, WIDE_NORM, EPI_STORE>(a, pieces, M, cu_count, n_blk, st);
    if (src == WIDE_NORM && epi == EPI_SWIGLU) return launch_wide_k<WT, WIDE_NORM, EPI_SWIGLU>(a, pieces, M, cu_count, n_blk, st);
    constexpr int F = std::is_same<WT, fp8e4m3>::value ? 2 : 1;          // a slice of 256 k per wave, or of 512
    if (src == WIDE_NORM_SUM && epi == EPI_SWIGLU && M == 1) {
        PGK_REQUIRE(a.nsplit >= 1 && a.nsplit <= 2 && a.part && a.h_out && a.h_out != a.h, "wide_proj: %d partial vectors", a.nsplit);
        if (a.K <= 2048) return launch_wide<WT, WIDE_NORM_SUM, EPI_SWIGLU, 2 / F, 1, 2>(a, pieces, M, cu_count, n_blk, st);
        return launch_wide<WT, WIDE_NORM_SUM, EPI_SWIGLU, 4 / F, 1, 2>(a, pieces, M, cu_count, n_blk, st);
    }
    if (src == WIDE_MERGE && epi == EPI_STORE && M == 1) {
        PGK_REQUIRE(a.nsplit >= 1 && wide_merge_ok(a.K, a.ld_out, a.nsplit) && a.part, "wide_proj: %d slices of heads of %d", a.nsplit, a.ld_out);
        return launch_wide<WT, WIDE_MERGE, EPI_STORE, 2 / F, 1, WIDE_SLICES>(a, pieces, M, cu_count, n_blk, st);
    }
    if (src == WIDE_PLAIN && epi == EPI_RESID) return launch_wide_k<WT, WIDE_PLAIN, EPI_RESID>(a, pieces, M, cu_count, n_blk, st);
    if (src == WIDE_PIECES && epi == EPI_RESID) return launch_wide_k<WT, WIDE_PIECES, EPI_RESID>(a, pieces, M, cu_count, n_blk, st);
    if constexpr (std::is_same<WT, bf16>::value) {
        if (src == WIDE_PLAIN && epi == EPI_STORE) return launch_wide_k<WT, WIDE_PLAIN, EPI_STORE>(a, pieces, M, cu_count, n_blk, st);
        if (src == WIDE_NORM && epi == EPI_LOGITS) return launch_wide_k<WT, WIDE_NORM, EPI_LOGITS>(a, pieces, M, cu_count, n_blk, st);
    }
    return set_error(PGK_ERR_INVALID, "wide_proj: source %d with epilogue %d", src, epi);
}

}  // namespace

bool wide_proj_ok(int N, int K, bool pieces) { return N >= 8 && N % 8 == 0 && K >= 256 && K % 256 == 0 && (pieces || K <= 4096); }

pgk_status wide_proj(bool fp8, int src, int epi, const FusedArgs& a, bf16* pieces, int M, int cu_count, int* n_blk, hipStream_t st) {
    PGK_REQUIRE(M >= 1 && M <= 8 && wide_proj_ok(a.N, a.K, src == WIDE_PIECES), "wide_proj: M %d N %d K %d", M, a.N, a.K);
    return fp8 ? launch_wide_e<fp8e4m3>(src, epi, a, pieces, M, cu_count, n_blk, st) : launch_wide_e<bf16>(src, epi, a, pieces, M, cu_count, n_blk, st);
}

}  // namespace pgk
