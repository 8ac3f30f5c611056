// Flash-attention prefill for gfx950 (bf16 / f16, head_dim 64 or 128), second generation.
//
// Orientation: the scores are computed TRANSPOSED, S^T[kv][q] = K . Q^T on v_mfma_f32_32x32x16, so a lane owns one
// query column (q = lane & 31) and its 16 accumulator registers per 32-kv sub-tile are kv rows.  Consequences:
//   * the online softmax (max, exp2, sum) of a query row is lane-local arithmetic over registers plus ONE exchange
//     with lane ^ 32 (the other half of the rows) - no LDS, no 16-lane butterflies;
//   * the probabilities are already laid out as the B operand of the second product O^T[d][q] += V^T[d][kv] . P^T[kv][q]:
//     registers 8s..8s+7 of a sub-tile, packed pairwise to 16-bit, ARE the k-step-s fragment (k order permuted:
//     element j of lane half h is kv = 16s + 8(j>>2) + 4h + (j&3)); the V^T operand is read in the same permuted
//     order out of V's row-major image by gfx950's transposing LDS read (two ds_read_b64_tr_b16 per fragment), so P
//     never touches LDS;
//   * the scores are scaled in fp32 under the exponential, exp2(s * scale - m): one fma where a subtraction would do (q used to
//     be multiplied by the scale before, which rounded it to 16 bits once more and was no faster);
//   * alpha (the running-max rescale) and 1/l are per-lane scalars for the O^T accumulators (q is again the lane).
// (V used to be transposed by a pass of its own over the whole context: 5.3 us of a 1531-token prompt's 42 us of
// attention per layer, 5.8 of 42 for 384 tokens at position 3201.)
// Workgroup = 4 waves (or two sides of 4, each with half the KV tiles: flash_plan) = 128 query rows of one head; KV tiles of 64 positions, K and V [64][D] double
// buffered in LDS (64 KiB at D = 128: two workgroups per CU), fetched by LDS-DMA, K a tile ahead of V: the products
// S(t + 1) run between the exponentials of S(t).  One barrier per tile.
// Workgroups are ordered heavy-first (causal: late query tiles see more keys) and all query heads of a kv head
// share id % Hkv, i.e. an XCD when Hkv is a multiple of 8, so the K/V stream of a head is served by one L2.
// Mask: kv_pos <= (kv_len - q_len) + q_pos  (reference: native/ops/nn/attention_kernels.cuh:32-148).

#include <algorithm>
#include <type_traits>

#include "flash.hip.h"
#include "flash_plan.h"
#include "latent.hip.h"
#include "pgk_device.hip.h"
#include "pgk_internal.h"

namespace pgk {

typedef __bf16 bf16x8_fl __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_fl __attribute__((ext_vector_type(8)));
typedef float f32x16_fl __attribute__((ext_vector_type(16)));

template <class T> __device__ __forceinline__ f32x16_fl mfma32(const uint4& a, const uint4& b, f32x16_fl c);
template <> __device__ __forceinline__ f32x16_fl mfma32<bf16>(const uint4& a, const uint4& b, f32x16_fl c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_fl, a), __builtin_bit_cast(bf16x8_fl, b), c, 0, 0, 0);
}
template <> __device__ __forceinline__ f32x16_fl mfma32<f16>(const uint4& a, const uint4& b, f32x16_fl c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_fl, a), __builtin_bit_cast(f16x8_fl, b), c, 0, 0, 0);
}
template <class T> __device__ __forceinline__ uint32_t pack16x2(float lo, float hi);
template <> __device__ __forceinline__ uint32_t pack16x2<bf16>(float lo, float hi) { return pack_bf16x2(lo, hi); }
template <> __device__ __forceinline__ uint32_t pack16x2<f16>(float lo, float hi) {
    return (uint32_t)__builtin_bit_cast(uint16_t, static_cast<_Float16>(lo)) | ((uint32_t)__builtin_bit_cast(uint16_t, static_cast<_Float16>(hi)) << 16);
}

struct FlashStrides { long long qh, qs, kh, ks, oh, os; };

// One wave-instruction of LDS-DMA: 64 lanes x 16 bytes at per-lane byte offsets of a buffer to LDS [lds, +1024), zeros beyond its end.  (Inline asm: for the
// builtin hipcc waits for the DMA in front of the next LDS read, whichever buffer that reads.  The waits are the explicit ones in the kernel.)
typedef uint32_t fl_u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void fl_dma16(const fl_u32x4& buffer, uint32_t off, uint32_t lds, int at) {
    asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(off), "s"(buffer), "s"(lds), "i"(at) : "memory", "m0", "scc");
}
__device__ __forceinline__ uint32_t fl_lds_addr(const char* p) { return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)p; }

constexpr int FL_THREADS = 256;
static_assert(FL_BQ == FLASH_ITEM_ROWS, "a listed query tile is one of the kernel's");

// K image: [64 kv][D] 16-bit, 16-byte chunk c (0..D/8-1) of row r at r*2D + ((c ^ (r & (D/8-1))) << 4)
template <int D> __device__ __forceinline__ int fl_k_off(int r, int c) { return r * (2 * D) + ((c ^ (r & (D / 8 - 1))) << 4); }
// V image: [64 kv][D] 16-bit, chunk c of row r at r*2D + ((c ^ x(r)) << 4).  A transposing read takes rows 4n .. 4n+3 (two n, by
// lane half), 64 contiguous bytes of each: x moves the four rows of an n into different 64-byte parts of the 256 bytes of banks.
template <int D> __device__ __forceinline__ int fl_v_sw(int r) { return D == 128 ? ((r & 3) << 2) | ((r >> 2) & 3) : (((r >> 1) & 1) << 2) | ((r >> 2) & 3); }
template <int D> __device__ __forceinline__ int fl_v_off(int r, int c) { return r * (2 * D) + ((c ^ fl_v_sw<D>(r)) << 4); }

// Several sequences in one launch (flash.hip.h): a workgroup takes one query tile of one of them instead of what its id says.
struct FlashMany {
    const FlashItem* items;
    int n_items, rows;             // rows: query rows of all sequences
    long long slot_stride;         // elements between the caches of two slots
};

// KV split: nsplit > 1 cuts a query tile's KV tiles into nsplit contiguous runs, one workgroup each; every workgroup leaves a
// NORMALISED partial output (type T) and its (m, l) per row, and flash_merge_kernel combines them.
struct FlashSplit {
    int nsplit;
    int run;        // > 0: KV tiles of a run, as many runs as a query tile's tiles make (at most nsplit)
    float* ml;      // [nsplit][Hq][q_len][2]  (m in the exp2 domain, l)
    void* o;        // [nsplit][q_len][Hq][D] of T, or of fp32 (`wide`: up to 128 query rows, and several sequences in one launch)
    bool wide;
    // fp8 x fp8 prefill (D = 128, bf16): instead of out, e4m3 codes [q_len][Hq * D] and one scale per (row, head) [q_len][Hq]
    // - a head's 128 output dims ARE one 128-wide scale block of the o_proj's A operand (quantize_fp8_rows' contract:
    // scale = absmax / 448 of the bf16-rounded values, 1 for an all-zero block), written by whichever kernel holds the final
    // row: this one (nsplit == 1) or flash_merge_kernel
    uint8_t* q8;
    float* q8s;
};

// Sliding window (WIN instantiations): query i sees keys i - window + 1 .. i, tiles left of a workgroup's first window are never
// loaded.  `gate`: OutGate, one value per (query row, head) or per element.
// BIAS instantiations: slopes[head] * (query - key) is taken off the scaled score - the accumulators of S = K . Q^T start at
// -slope / scale * (query - key) instead of zero.
struct FlashWindow {
    int window;
    OutGate gate;
    const float* slopes;
    float inv_scale;
};
template <class T> __device__ __forceinline__ float flash_gate(const FlashWindow& w, int qrow, int head) {
    if (!w.gate.p || w.gate.gc) return 1.f;
    return 1.0f / (1.0f + __expf(-to_f(reinterpret_cast<const T*>(w.gate.p)[(long long)qrow * w.gate.gs + head * w.gate.gh])));
}
// the elementwise form: N consecutive columns (aligned to N elements) from column c on
template <class T, int N> __device__ __forceinline__ void flash_gate_cols(const FlashWindow& w, int qrow, int head, int c, float (&y)[N]) {
    const T* g = reinterpret_cast<const T*>(w.gate.p) + (long long)qrow * w.gate.gs + head * w.gate.gh + c;
    uint2 raw[N / 4];
#pragma unroll
    for (int j = 0; j < N / 4; ++j) raw[j] = *reinterpret_cast<const uint2*>(g + 4 * j);
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const uint32_t word = j & 2 ? raw[j / 4].y : raw[j / 4].x;
        const uint16_t half = (uint16_t)(j & 1 ? word >> 16 : word);
        y[j] /= 1.0f + __expf(-to_f(__builtin_bit_cast(T, half)));
    }
}

template <class T, int D, bool WIN = false, bool BIAS = false, int SIDES = 1>
__global__ __launch_bounds__(SIDES * FL_THREADS, D == 64 && WIN ? 3 : 2) void flash_fwd_kernel(const T* q, const T* k, const T* v, T* out, int hq, int hkv,
                                                              int q_len, int kv_len, float scale_log2e, FlashStrides sd,
                                                              FlashSplit sp, FlashWindow win, FlashMany many) {
    constexpr int NC = D / 8;            // 16-byte chunks per K row
    constexpr int KS = D / 16;           // k-steps of Q.K^T
    constexpr int DT = D / 32;           // 32-row tiles of O^T
    constexpr int K_BYTES = 64 * D * 2, V_BYTES = K_BYTES;
    extern __shared__ __attribute__((aligned(16))) char fl_smem[];   // of each side K[2] | V[2]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wid = wave & 3, ql = lane & 31, h = lane >> 5;
    const int side = SIDES == 1 ? 0 : wave >> 2, side_at = side * (2 * K_BYTES + 2 * V_BYTES);

    // workgroup id -> (kv head, query head in its group, query tile, KV run), heavy tiles first
    const int rep = hq / hkv;
    const int id = blockIdx.x;
    const int kvh = id % hkv, rest = id / hkv;
    const int head = kvh * rep + rest % rep;
    const int rest2 = rest / rep;
    int split, qt, row0 = 0, rows = q_len, nsplit = sp.nsplit;
    if (many.items) {
        const FlashItem it = many.items[rest2 / sp.nsplit];
        split = rest2 % sp.nsplit;
        row0 = __builtin_amdgcn_readfirstlane(it.row0);
        q_len = __builtin_amdgcn_readfirstlane(it.q_len);
        kv_len = __builtin_amdgcn_readfirstlane(it.kv_len);
        const int st = __builtin_amdgcn_readfirstlane(it.slot_tile);
        qt = st & 0xFFFF;
        rows = many.rows;
        q += (long long)row0 * sd.qs;
        out += (long long)row0 * sd.os;
        k += (st >> 16) * many.slot_stride;
        v += (st >> 16) * many.slot_stride;
    } else if (!WIN && sp.run > 0) {
        qt = (q_len + FL_BQ - 1) / FL_BQ - 1;
        split = rest2;
        for (nsplit = flash_runs(qt, q_len, kv_len, sp.run); split >= nsplit; nsplit = flash_runs(--qt, q_len, kv_len, sp.run)) split -= nsplit;
    } else {
        // heavy tiles first - and, when the launch is one round of two workgroups per CU (KV split), the second half of the ids in
        // ASCENDING weight: a CU's two residents are then a heavy and a light run (ids i and i + grid / 2 sit on the same CU when
        // the dispatcher deals one workgroup to every CU before the second)
        const int nqt = (q_len + FL_BQ - 1) / FL_BQ, nord = nqt * sp.nsplit;
        int order = rest2;
        if (sp.nsplit > 1 && order >= nord / 2) order = nord / 2 + (nord - 1 - order);
        split = order % sp.nsplit;
        qt = nqt - 1 - order / sp.nsplit;
    }
    const int qw0 = qt * FL_BQ + wid * 32;          // first query row of this wave
    const int causal_off = kv_len - q_len;
    const T* qh = q + (size_t)head * sd.qh;
    const T* kh = k + (size_t)kvh * sd.kh;
    const T* vh = v + (size_t)kvh * sd.kh;

    uint4 qf[KS];
    f32x16_fl o[DT];
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[i][r] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;    // running max (scaled, log2 domain) and this lane's half of the row sum

    const int q_last = min(qt * FL_BQ + FL_BQ - 1, q_len - 1);
    const int kv_end = min(kv_len, causal_off + q_last + 1);
    const int nt_all = (kv_end + FL_BKV - 1) / FL_BKV;
    // this workgroup's run of KV tiles [t0, t1)
    const int first_kv = WIN ? causal_off + qt * FL_BQ - win.window + 1 : 0;
    const int tb = WIN && first_kv > 0 ? first_kv / FL_BKV : 0;            // tiles before it are outside every row's window
    int t0 = tb + (int)((long long)(nt_all - tb) * split / nsplit), t1 = tb + (int)((long long)(nt_all - tb) * (split + 1) / nsplit);
    int last = t1;                                  // where the loop ends; both sides pass as many barriers
    if constexpr (SIDES == 2) {
        const int half = (t1 - t0 + 1) / 2;
        if (side) t0 += half;
        else t1 = t0 + half;
        last = t0 + half;
    }

    // One wave-instruction of LDS-DMA moves 1 KiB = ROWS rows; the images' swizzles are applied on the source side (lane l of a row fetches the chunk that belongs
    // into its 16 bytes).  A wave moves NI instructions of K and of V per tile.  A tile is a buffer of the rows that are there: what lies beyond comes as zeros
    // without a branch (their probabilities are zero too), and a tile past the run's end reads nothing.
    constexpr int ROWS = 64 / NC, NI = 64 / ROWS / 4;
    const int dr = lane / NC, ds = lane % NC;
    uint32_t ko[NI], vo[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int r = wid * 16 + i * ROWS + dr;
        ko[i] = (uint32_t)(r * sd.ks + (ds ^ (r & (NC - 1))) * 8) * 2;
        vo[i] = (uint32_t)(r * sd.ks + (ds ^ fl_v_sw<D>(r)) * 8) * 2;
    }
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(fl_lds_addr(fl_smem) + side_at + wid * NI * 1024), row_bytes = (uint32_t)(sd.ks * 2);
    const uint64_t tile_bytes = (uint64_t)sd.ks * (FL_BKV * 2);
    const int kv_stop = min(kv_len, t1 * FL_BKV);
    auto bytes_of = [&](int t) { const int n = min(kv_stop - t * FL_BKV, FL_BKV); return n > 0 ? (n - 1) * row_bytes + 2 * D : 0u; };
    auto tile_at = [&](uint64_t at, uint32_t bytes) { return fl_u32x4{(uint32_t)at, (uint32_t)(at >> 32) & 0xFFFFu, bytes, 0x00020000u}; };   // raw, 32-bit words
    uint64_t k_at = (uint64_t)(uintptr_t)kh + t0 * tile_bytes, v_at = (uint64_t)(uintptr_t)vh + t0 * tile_bytes;       // where the next DMA reads
    auto dma_k = [&](int buf, uint32_t bytes) {
        const fl_u32x4 tile = tile_at(k_at, bytes);
#pragma unroll
        for (int i = 0; i < NI; ++i) fl_dma16(tile, ko[i], lds0, buf * K_BYTES + i * 1024);
        k_at += tile_bytes;
    };
    auto dma_v = [&](int buf, uint32_t bytes) {
        const fl_u32x4 tile = tile_at(v_at, bytes);
#pragma unroll
        for (int i = 0; i < NI; ++i) fl_dma16(tile, vo[i], lds0, 2 * K_BYTES + buf * V_BYTES + i * 1024);
        v_at += tile_bytes;
    };
    // S^T = K . Q^T of one tile: two 32-kv sub-tiles (rows = positions, column = this lane's query)
    // Windows of head dim 64 hold one register for the mask's two ends and the bias (a row that is there sees none behind the context): with three the kernel with slopes takes 189, of which a SIMD holds two
    // waves and not three.  16 heads, 1500 rows, 1024 positions, us, 189 / 168: 28.1 / 23.7; 32 heads 36.3 / 30.7.  (Head dim 128 holds two anyway and is 0.5 % faster with three.)
    constexpr bool FEW = WIN && D == 64;
    const int q_at = FEW ? causal_off + qw0 + ql - 4 * h : 0;
    const float slope = BIAS ? win.slopes[head] * win.inv_scale : 0.f;
    auto s_init = [&](int t, f32x16_fl& s0, f32x16_fl& s1) {
        if constexpr (BIAS) {            // rows are keys kv0 + (r & 3) + 8 (r >> 2) + 4 h (+ 32), this lane's query is position q_at + 4 h
            const float b0 = slope * (float)(FEW ? t * FL_BKV - q_at : t * FL_BKV + 4 * h - (causal_off + qw0 + ql));
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                s0[r] = fmaf(slope, (float)((r & 3) + 8 * (r >> 2)), b0);
                s1[r] = fmaf(slope, (float)(32 + (r & 3) + 8 * (r >> 2)), b0);
            }
        } else {
#pragma unroll
            for (int r = 0; r < 16; ++r) { s0[r] = 0.f; s1[r] = 0.f; }
        }
    };
    const char* ka[KS];                  // of the first buffer and sub-tile
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) ka[ks] = fl_smem + side_at + fl_k_off<D>(ql, 2 * ks + h);
    auto k_frag = [&](int buf, int half, int ks) { return *reinterpret_cast<const uint4*>(ka[ks] + buf * K_BYTES + half * 64 * D); };
    // tiles entirely above this wave's diagonal contribute nothing (wave-uniform)
    auto live = [&](int t) -> bool {
        return t < t1 && t * FL_BKV <= causal_off + qw0 + 31 && (!WIN || t * FL_BKV + FL_BKV - 1 > causal_off + qw0 - win.window);
    };

    // One KV tile per iteration: softmax of S(t) with the products S(t + 1) = K(t + 1) . Q^T between its exponentials - in one basic block, a matrix instruction
    // behind every two of them - then O += V(t) . P.  So K runs a tile ahead of V: the DMA of K(t + 2) and V(t + 1) goes out behind the barrier at which K(t + 1)
    // and V(t) have landed and S(t) and O(t - 1) have been read.  Attention with merge, us, staged through registers with S(t) in front of its softmax / this: 16
    // heads, 1531 rows 35.4 / 30.6, 384 at 3585 34.0 / 29.0; 32 heads, 4096 rows 180 / 151.  (As two conditional blocks hipcc keeps S(t + 1) and the softmax apart; the
    // DMA a piece behind each k-step, inside the block, spills 74 registers.)
    // A pass of the loop is two tiles: the buffers' places are immediates then, and S(t + 1) is not copied.  V is read a k-step ahead of its products (the first under the last of S), the first of K
    // above the softmax; the row sums and the next tile's largest scores are taken under the products with V, where only the matrix units had work, and waves there go first (s_setprio): two on a
    // SIMD otherwise meet in the same phase.  Before / with all of it, us: 16 heads, 1531 rows 29.7 / 27.7, 384 at 3585 30.2 / 27.8, 400 13.4 / 11.9, 2500 52.2 / 45.2; 32 heads, 1000 rows 26.4 / 23.9,
    // 4096 171 / 143 (of it s_setprio 155 / 143; 3000 rows 88.6 / 83.6).  A tile was 270 vector instructions beside 32 matrix instructions, of which two waves overlapped a tenth.
    // (As a lambda called for both tiles the windows' kernels spill 70 registers.)
    constexpr bool AHEAD = !WIN;         // V, sums and scores: windows have no registers for it
    f32x16_fl sc[2][2];                  // S of a pass's two tiles
    dma_k(0, bytes_of(t0));
    uint32_t v_bytes = bytes_of(t0 + 1);
    dma_k(1, v_bytes);
    dma_v(0, bytes_of(t0));
    // Q^T fragments (B operand): lane = query column, k = d
    {
        const T* qrow = qh + (size_t)min(qw0 + ql, q_len - 1) * sd.qs + 8 * h;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) qf[ks] = *reinterpret_cast<const uint4*>(qrow + ks * 16);
    }
    // Retire the Q loads (and with them the first tiles) HERE: still counted as pending at the loop header, they would be waited for in every iteration, behind
    // the DMA that it has just issued.
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) asm volatile("" ::"v"(qf[ks].x), "v"(qf[ks].y), "v"(qf[ks].z), "v"(qf[ks].w));
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    s_init(t0, sc[0][0], sc[0][1]);
    if (live(t0)) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            sc[0][0] = mfma32<T>(k_frag(0, 0, ks), qf[ks], sc[0][0]);
            sc[0][1] = mfma32<T>(k_frag(0, 1, ks), qf[ks], sc[0][1]);
        }
    }
    // V^T fragments: lane l gets dim 32 i + (l & 31) of rows 16 s + 8 u + 4 h .. + 3.  A 16-lane group's transposing read covers 4 rows x 16
    // dims: lane l15 of it supplies the address of row l15 >> 2, dims 4 (l15 & 3) .. + 3.  The swizzle of such a row depends on l15 >> 2, h and
    // u only, so the addresses of (i, u) serve every s with an immediate offset of 16 rows.
    typedef short fl_v4s __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) fl_v4s* fl_lds_v4;
    const int tr = (lane & 15) >> 2, tc = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1), t8 = 8 * (lane & 1);
    const char* va[DT][2];
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
        for (int u = 0; u < 2; ++u) va[i][u] = fl_smem + side_at + 2 * K_BYTES + fl_v_off<D>(8 * u + 4 * h + tr, 4 * i + tc) + t8;
    auto v_frag = [&](int buf, int i, int u, int s) {
        return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((fl_lds_v4)(va[i][u] + buf * V_BYTES + s * 32 * D)));
    };
    // this lane's largest score, in two chains of v_max3_f32
    auto largest = [&](const f32x16_fl& a, const f32x16_fl& b) -> float {
        float x = -INFINITY, y = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
            x = fmaxf(fmaxf(x, a[r]), a[r + 1]);
            y = fmaxf(fmaxf(y, b[r]), b[r + 1]);
        }
        return fmaxf(x, y);
    };
    // ... and the row's (the other half of it is in lane ^ 32), in the log2 domain: -inf stays -inf (scale > 0)
    auto scaled = [&](float x) -> float {
        const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
        return fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1])) * scale_log2e;
    };
    float top = -INFINITY;               // of S(t), before a mask
    if constexpr (AHEAD) top = scaled(largest(sc[0][0], sc[0][1]));
    // tile t: sc0 | sc1 are S(t), sn0 | sn1 become S(t + 1); V(t) is in buffer buf, K(t + 1) in the other
    for (int t2 = t0; t2 < last; t2 += 2)
#pragma unroll
    for (int buf = 0; buf < 2; ++buf) {
        const int t = t2 + buf, kv0 = t * FL_BKV;
        if (buf && t == last) break;
        f32x16_fl &sc0 = sc[buf][0], &sc1 = sc[buf][1], &sn0 = sc[buf ^ 1][0], &sn1 = sc[buf ^ 1][1];
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                 // this wave's share of K(t + 1) and V(t)
        __syncthreads();                                                 // ... everyone's; and everyone has read K(t) and V(t - 1)
        const uint32_t k_bytes = bytes_of(t + 2);
        dma_k(buf, k_bytes);
        dma_v(buf ^ 1, v_bytes);
        v_bytes = k_bytes;
        if (live(t)) {                                                   // (behind the last tile, S(t + 1) is of what K's other buffer holds, and unused)
            uint4 k0 = k_frag(buf ^ 1, 0, 0), k1 = k_frag(buf ^ 1, 1, 0);
            // ---- mask, online softmax (this lane: query qw0 + ql, kv rows (r&3) + 8(r>>2) + 4h of each sub-tile) ----
            const bool need_mask = kv0 + FL_BKV - 1 > causal_off + qw0 || kv0 + FL_BKV > kv_len ||
                                   (WIN && kv0 <= causal_off + qw0 + 31 - win.window);   // wave-uniform
            const int lim = FEW ? q_at - kv0 : min(causal_off + qw0 + ql, kv_len - 1) - kv0 - 4 * h;                    // local kv row <= lim is visible
            const int low = !WIN ? 0 : FEW ? lim - win.window + 1 : causal_off + qw0 + ql - win.window + 1 - kv0 - 4 * h;       // ... and >= low with a window
            float mx = top;
            if (need_mask) {   // diagonal / ragged tiles only: a real wave-uniform branch, not 32 predicated selects per tile
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int kvl = (r & 3) + 8 * (r >> 2);
                    sc0[r] = kvl <= lim && (!WIN || kvl >= low) ? sc0[r] : -INFINITY;
                    sc1[r] = 32 + kvl <= lim && (!WIN || 32 + kvl >= low) ? sc1[r] : -INFINITY;
                }
            }
            if (!AHEAD || need_mask) mx = scaled(largest(sc0, sc1));
            // Deferred rescale: the reference point of a row only moves when its maximum grew by more than 6 (log2
            // domain), so probabilities stay <= 64 (exact in fp32 sums, fine in 16-bit P) and on most tiles - for the whole
            // wave - alpha is exactly 1 and the 64-multiply rescale of O is skipped.
            const float m_new = (mx > m_run + 6.0f || m_run == -INFINITY) ? fmaxf(m_run, mx) : m_run;
            const float m_use = m_new == -INFINITY ? 0.f : m_new;        // a fully masked row so far: p = exp2(-inf) = 0
            const bool moved = __builtin_amdgcn_ballot_w64(m_new != m_run) != 0;   // wave-uniform
            const float alpha = moved ? __builtin_amdgcn_exp2f(m_run - m_use) : 1.0f;   // m_run = -inf -> 0 (accumulators are 0 anyway)
            if (moved) {                                                 // (in front of the block below, which it would cut in two)
#pragma unroll
                for (int i = 0; i < DT; ++i)
#pragma unroll
                    for (int r = 0; r < 16; ++r) o[i][r] *= alpha;
            }
            uint4 vf[2][DT];                                             // V, a k-step ahead of its products
            auto load_v = [&](int s) {
#pragma unroll
                for (int i = 0; i < DT; ++i) {
                    const uint2 lo = v_frag(buf, i, 0, s), hi = v_frag(buf, i, 1, s);
                    vf[s & 1][i] = make_uint4(lo.x, lo.y, hi.x, hi.y);
                }
            };
            float ls0 = 0.f, ls1 = 0.f, tx = -INFINITY, ty = -INFINITY;
            uint32_t pw0[8], pw1[8];                                     // P, packed
            s_init(t + 1, sn0, sn1);
            __builtin_amdgcn_sched_barrier(0);
            constexpr int PER = 16 / KS;                                 // rows of S(t) per k-step of S(t + 1)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                const uint4 n0 = k_frag(buf ^ 1, 0, ks + 1 < KS ? ks + 1 : ks), n1 = k_frag(buf ^ 1, 1, ks + 1 < KS ? ks + 1 : ks);
                if (AHEAD && ks == KS - 1) load_v(0);
                sn0 = mfma32<T>(k0, qf[ks], sn0);
#pragma unroll
                for (int r = ks * PER; r < (ks + 1) * PER; ++r) {
                    sc0[r] = __builtin_amdgcn_exp2f(fmaf(sc0[r], scale_log2e, -m_use));
                    sc1[r] = __builtin_amdgcn_exp2f(fmaf(sc1[r], scale_log2e, -m_use));
                    if (!AHEAD) ls0 += sc0[r], ls1 += sc1[r];
                    if (r == ks * PER + PER / 2 - 1) sn1 = mfma32<T>(k1, qf[ks], sn1);
                }
#pragma unroll
                for (int r = ks * PER; r < (ks + 1) * PER; r += 2) {
                    pw0[r / 2] = pack16x2<T>(sc0[r], sc0[r + 1]);
                    pw1[r / 2] = pack16x2<T>(sc1[r], sc1[r + 1]);
                }
                k0 = n0;
                k1 = n1;
                __builtin_amdgcn_sched_barrier(0);
            }
            m_run = m_new;
            // ---- O^T += V^T . P^T : 4 k-steps of 16 kv ----
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const uint32_t* w = s < 2 ? pw0 + 4 * s : pw1 + 4 * (s - 2);
                const uint4 pb = make_uint4(w[0], w[1], w[2], w[3]);
                if (!AHEAD) load_v(s);
                else if (s < 3) load_v(s + 1);
                if (AHEAD) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < DT; ++i) o[i] = mfma32<T>(vf[s & 1][i], pb, o[i]);
                // the matrix units have work: the sums, and the next tile's largest score
#pragma unroll
                for (int r = 4 * s; AHEAD && r < 4 * s + 4; ++r) ls0 += sc0[r], ls1 += sc1[r];
                if (AHEAD && (s == 1 || s == 2)) {
#pragma unroll
                    for (int r = 8 * (s - 1); r < 8 * s; r += 2) {
                        tx = fmaxf(fmaxf(tx, sn0[r]), sn0[r + 1]);
                        ty = fmaxf(fmaxf(ty, sn1[r]), sn1[r + 1]);
                    }
                }
                if (AHEAD && s == 3) top = scaled(fmaxf(tx, ty));
                if (AHEAD) __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_s_setprio(0);
            l_run = l_run * alpha + (ls0 + ls1);
        } else {
            if (WIN && live(t + 1)) {                                    // left of this wave's windows: the next tile's scores alone
                s_init(t + 1, sn0, sn1);
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    sn0 = mfma32<T>(k_frag(buf ^ 1, 0, ks), qf[ks], sn0);
                    sn1 = mfma32<T>(k_frag(buf ^ 1, 1, ks), qf[ks], sn1);
                }
            }
        }
    }

    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                     // requests past the run's end, before the LDS is given back
    if constexpr (SIDES == 2) {      // the second side's state comes to the first by way of the tiles' place
        __syncthreads();
        float4* mine = reinterpret_cast<float4*>(fl_smem) + wid * (4 * DT + 1) * 64 + lane;
        if (side) {
#pragma unroll
            for (int i = 0; i < DT; ++i)
#pragma unroll
                for (int g = 0; g < 4; ++g) mine[(4 * i + g) * 64] = make_float4(o[i][4 * g], o[i][4 * g + 1], o[i][4 * g + 2], o[i][4 * g + 3]);
            mine[4 * DT * 64] = make_float4(m_run, l_run, 0.f, 0.f);
        }
        __syncthreads();
        if (side) return;
        const float4 ml = mine[4 * DT * 64];
        const float m = fmaxf(m_run, ml.x), m_use = m == -INFINITY ? 0.f : m;
        const float a0 = __builtin_amdgcn_exp2f(m_run - m_use), a1 = __builtin_amdgcn_exp2f(ml.x - m_use);
        l_run = l_run * a0 + ml.y * a1;
        m_run = m;
#pragma unroll
        for (int i = 0; i < DT; ++i)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const float4 v = mine[(4 * i + g) * 64];
                o[i][4 * g] = fmaf(v.x, a1, o[i][4 * g] * a0);
                o[i][4 * g + 1] = fmaf(v.y, a1, o[i][4 * g + 1] * a0);
                o[i][4 * g + 2] = fmaf(v.z, a1, o[i][4 * g + 2] * a0);
                o[i][4 * g + 3] = fmaf(v.w, a1, o[i][4 * g + 3] * a0);
            }
    }

    // ---- normalise and store: lane = query row, registers 4g..4g+3 of tile i are d = 32i + 8g + 4h .. +3 ----
    const float l_tot = l_run + __shfl_xor(l_run, 32, 64);
    float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
    const int qrow = qw0 + ql;
    if constexpr (WIN) { if (nsplit == 1) inv *= flash_gate<T>(win, min(qrow, q_len - 1), head); }
    if constexpr (std::is_same<T, bf16>::value && D == 128) {
        if (sp.q8 != nullptr && nsplit == 1) {       // workgroup-uniform
            // the lane's 64 dims (the partner lane ^ 32 holds the other 64), rounded to bf16 as the plain store would
            float amax = 0.f;
#pragma unroll
            for (int i = 0; i < DT; ++i)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    o[i][e] = __uint_as_float(pack_bf16x2(o[i][e] * inv, 0.f) << 16);
                    amax = fmaxf(amax, fabsf(o[i][e]));
                }
            amax = fmaxf(amax, __shfl_xor(amax, 32, 64));
            const float sc = amax > 0.f ? amax / 448.0f : 1.0f;
            if (qrow < q_len) {
                uint8_t* qrow8 = sp.q8 + ((size_t)(row0 + qrow) * hq + head) * D;
#pragma unroll
                for (int i = 0; i < DT; ++i)
#pragma unroll
                    for (int g = 0; g < 4; ++g)
                        *reinterpret_cast<uint32_t*>(qrow8 + i * 32 + 8 * g + 4 * h) =
                            pack_fp8x4(o[i][4 * g] / sc, o[i][4 * g + 1] / sc, o[i][4 * g + 2] / sc, o[i][4 * g + 3] / sc);
                if (h == 0) sp.q8s[(size_t)(row0 + qrow) * hq + head] = sc;
            }
            return;
        }
    }
    if (qrow < q_len) {
        float* wrow = nsplit > 1 && sp.wide ? reinterpret_cast<float*>(sp.o) + (((size_t)split * rows + row0 + qrow) * hq + head) * D : nullptr;
        T* orow = nsplit > 1 ? reinterpret_cast<T*>(sp.o) + (((size_t)split * rows + row0 + qrow) * hq + head) * D
                                : out + (size_t)head * sd.oh + (size_t)qrow * sd.os;
#pragma unroll
        for (int i = 0; i < DT; ++i)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                float y[4] = {o[i][4 * g] * inv, o[i][4 * g + 1] * inv, o[i][4 * g + 2] * inv, o[i][4 * g + 3] * inv};
                if constexpr (WIN) { if (win.gate.gc && nsplit == 1) flash_gate_cols<T, 4>(win, qrow, head, i * 32 + 8 * g + 4 * h, y); }
                if (wrow) *reinterpret_cast<float4*>(wrow + i * 32 + 8 * g + 4 * h) = make_float4(y[0], y[1], y[2], y[3]);
                else *reinterpret_cast<uint2*>(orow + i * 32 + 8 * g + 4 * h) = make_uint2(pack16x2<T>(y[0], y[1]), pack16x2<T>(y[2], y[3]));
            }
        if (nsplit > 1 && h == 0) {
            float* ml = sp.ml + (((size_t)split * hq + head) * rows + row0 + qrow) * 2;
            ml[0] = m_run;
            ml[1] = l_tot;
        }
    }
}

// out[q][head][:] = sum_s w_s o_s / sum_s w_s,  w_s = l_s 2^(m_s - max m): one thread per 8 output elements.  Short work behind one round trip to memory:
// all records and the first RUNS partial rows are requested before anything is waited for (RUNS = 2, 4 or 8, whichever holds nsplit; beyond 8 runs,
// at most 16, the others follow).  The maximum used to be found in a round trip of its own, two runs asked for four
// rows, and the row and head of a thread were a 64-bit division: Qwen3-0.6B, 28 layers, us, before and after: 1531 rows 2988 / 2949, 384 rows at 3201 2175 / 2128,
// 100 at 2000 1450 / 1410, 1000 at 3000 3123 / 3090.
template <class T, class P, int D, int RUNS>   // P: type of the partial rows
__global__ __launch_bounds__(256) void flash_merge_kernel(const float* ml, const P* po, T* out, int hq, int q_len, int nsplit, long long oh, long long os,
                                                          uint8_t* q8 = nullptr, float* q8s = nullptr, FlashWindow win = FlashWindow{}, int run = 0, int kv_len = 0) {
    constexpr int CPR = D / 8, RECS = RUNS == 8 ? 16 : RUNS;
    const uint32_t gid = blockIdx.x * 256u + threadIdx.x, rowi = gid / CPR;      // several runs: at most two workgroups of 128 rows to a CU (flash_plan)
    if (rowi >= (uint32_t)q_len * hq) return;          // the 16 lanes of a (row, head) stay together
    const int c = (int)(gid % CPR), qrow = (int)(rowi / (uint32_t)hq), head = (int)(rowi % (uint32_t)hq);
    if (run > 0) {
        nsplit = flash_runs(qrow / FL_BQ, q_len, kv_len, run);
        if (nsplit == 1) return;                       // the run has left the row itself
    }
    uint4 v[RUNS][sizeof(P) / 2];
    float2 r[RECS];
    auto rows = [&](int s0) {
#pragma unroll
        for (int u = 0; u < RUNS; ++u)
#pragma unroll
            for (int x = 0; x < (int)sizeof(P) / 2; ++x)
                v[u][x] = *reinterpret_cast<const uint4*>(po + (((size_t)min(s0 + u, nsplit - 1) * q_len + qrow) * hq + head) * D + c * 8 + 4 * x);
    };
#pragma unroll
    for (int u = 0; u < RECS; ++u) r[u] = *reinterpret_cast<const float2*>(ml + (((size_t)min(u, nsplit - 1) * hq + head) * q_len + qrow) * 2);
    rows(0);
    float mstar = -INFINITY;
#pragma unroll
    for (int u = 0; u < RECS; ++u) mstar = fmaxf(mstar, r[u].x);       // (beyond nsplit the last one again)
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, den = 0.f;
#pragma unroll
    for (int s0 = 0; s0 < RECS; s0 += RUNS) {
        if (s0 > 0) {
            if (s0 >= nsplit) break;
            rows(s0);
        }
#pragma unroll
        for (int u = 0; u < RUNS; ++u) {
            // a run that saw no key has l = 0; any other counts, also one whose l is NaN
            const bool live = s0 + u < nsplit && __float_as_uint(r[s0 + u].y) != 0u;
            const float w = live ? r[s0 + u].y * __builtin_amdgcn_exp2f(r[s0 + u].x - mstar) : 0.f;
            float f[8];
            if constexpr (sizeof(P) == 4) {
#pragma unroll
                for (int x = 0; x < 2; ++x) {
                    f[4 * x] = __uint_as_float(v[u][x].x); f[4 * x + 1] = __uint_as_float(v[u][x].y);
                    f[4 * x + 2] = __uint_as_float(v[u][x].z); f[4 * x + 3] = __uint_as_float(v[u][x].w);
                }
            } else {
                Vec<P> t;
                t.raw = v[u][0];
                t.to_float(f);
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[j] = live ? fmaf(w, f[j], acc[j]) : acc[j];
            den += w;
        }
    }
    const float inv = (den > 0.f ? 1.f / den : 0.f) * flash_gate<T>(win, qrow, head);
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] *= inv;
    if (win.gate.gc) flash_gate_cols<T, 8>(win, qrow, head, c * 8, acc);
    Vec<T> y;
    y.from_float(acc);
    if constexpr (std::is_same<T, bf16>::value && D == 128) {
        if (q8 != nullptr) {                // see FlashSplit::q8: 16 lanes x 8 dims = one (row, head) = one scale block
            y.to_float(acc);
            float amax = 0.f;
#pragma unroll
            for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(acc[j]));
            amax = group16_max(amax);
            const float sc = amax > 0.f ? amax / 448.0f : 1.0f;
            uint2 o8;
            o8.x = pack_fp8x4(acc[0] / sc, acc[1] / sc, acc[2] / sc, acc[3] / sc);
            o8.y = pack_fp8x4(acc[4] / sc, acc[5] / sc, acc[6] / sc, acc[7] / sc);
            *reinterpret_cast<uint2*>(q8 + rowi * D + c * 8) = o8;
            if (c == 0) q8s[rowi] = sc;
            return;
        }
    }
    y.store(out + (size_t)head * oh + (size_t)qrow * os + c * 8);
}

static int flash_cus() {
    int dev = 0, cus = 0;
    return hipGetDevice(&dev) == hipSuccess && hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && cus > 0 ? cus : 256;
}

// q_len: query rows of all sequences where `many` lists several (kv_len: the longest context among them)
template <class T, int D, bool WIN = false, bool BIAS = false>
static pgk_status flash_launch(const T* q, const T* k, const T* v, T* out, int hq, int hkv, int q_len, int kv_len, float scale,
                               const FlashStrides& sd, hipStream_t st, uint8_t* q8 = nullptr, float* q8s = nullptr, const FlashWindow& win = FlashWindow{},
                               const FlashMany& many = FlashMany{}, bool one_side = false) {
    const int tiles = many.items ? many.n_items : ceil_div(q_len, FL_BQ), cus = flash_cus();
    const int span = WIN && (long long)win.window + FL_BQ < kv_len ? win.window + FL_BQ : kv_len;    // keys the heaviest query tile walks
    const FlashPlan even = WIN ? FlashPlan{flash_window_runs(cus, (long long)tiles * hq, span), 1, false, 0} : flash_even_plan(cus, (long long)tiles * hq, q_len, kv_len, 16);
    FlashPlan plan = WIN || many.items || one_side ? even : flash_plan(cus, even, hq, q_len, kv_len, D, 16);
    const bool wide = many.items || q_len <= 128 || plan.fp32;
    // Up to 128 rows need no scratch memory to be captured: one run (16 heads, us: 64 rows of 1000 31, 128 of 400 19, 100 of 4000 101; on the 64-row
    // tiles of the first-generation kernel 61, 31 and 239)
    if (plan.runs > 1 && q_len <= 128) {
        hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(st, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone) plan.runs = 1;
    }
    void* ws = nullptr;
    size_t ml_at = 0;
    plan = flash_granted(plan, even, [&](int runs) {      // no memory, or a stream whose end the pool cannot see: slower, and right
        ml_at = ((size_t)runs * q_len * hq * D * (wide ? 4 : sizeof(T)) + 255) & ~(size_t)255;
        return pool_malloc_on(&ws, ml_at + (size_t)runs * hq * q_len * 2 * sizeof(float), st) == PGK_OK;
    });
    const int nsplit = plan.runs;
    const FlashSplit sp{nsplit, plan.run, nsplit > 1 ? (float*)((char*)ws + ml_at) : nullptr, ws, wide, q8, q8s};
    auto launch = [&](auto sides) -> hipError_t {
        constexpr int SIDES = decltype(sides)::value;
        constexpr size_t LDS = SIDES * 4 * (size_t)(64 * D * 2);
        auto kernel = &flash_fwd_kernel<T, D, WIN, BIAS, SIDES>;
        static bool attr_done = false;
        if (LDS > 48 * 1024 && !attr_done) {
            if (hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS); e != hipSuccess) return e;
            attr_done = true;
        }
        int wgs = tiles * nsplit;
        if (sp.run > 0) {
            wgs = 0;
            for (int i = 0; i < tiles; ++i) wgs += flash_runs(i, q_len, kv_len, sp.run);
        }
        kernel<<<wgs * hq, SIDES * FL_THREADS, LDS, st>>>(q, k, v, out, hq, hkv, q_len, kv_len, scale * 1.4426950408889634f, sd, sp, win, many);
        return hipGetLastError();
    };
    hipError_t e;
    if constexpr (WIN) e = launch(std::integral_constant<int, 1>{});
    else e = plan.sides == 2 && !one_side ? launch(std::integral_constant<int, 2>{}) : launch(std::integral_constant<int, 1>{});
    if (e == hipSuccess && nsplit > 1) {
        const size_t work = (size_t)q_len * hq * (D / 8);
        const unsigned grid = (unsigned)((work + 255) / 256);
        auto merge = [&](auto* part, auto runs) {
            using P = std::remove_pointer_t<decltype(part)>;
            flash_merge_kernel<T, P, D, decltype(runs)::value><<<grid, 256, 0, st>>>(sp.ml, (const P*)part, out, hq, q_len, nsplit, sd.oh, sd.os, q8, q8s, win, sp.run, kv_len);
        };
        auto pick = [&](auto* part) {
            if (nsplit <= 2) merge(part, std::integral_constant<int, 2>{});
            else if (nsplit <= 4) merge(part, std::integral_constant<int, 4>{});
            else merge(part, std::integral_constant<int, 8>{});
        };
        if (wide) pick((float*)sp.o);
        else pick((T*)sp.o);
        e = hipGetLastError();
    }
    if (ws) pgk_free(ws);   // st's again: whatever takes it runs after the kernels above
    PGK_CHECK_HIP(e);
    return PGK_OK;
}

// entry used by ops_attention.hip's dispatcher and by an engine whose next step rounds the result to e4m3 (one_side); dt16: 0 = bf16, 1 = f16
pgk_status flash_prefill(const void* q, const void* k, const void* v, void* out, int hq, int hkv, int q_len, int kv_len, int d,
                         float scale, long long qh, long long qs, long long kh, long long ks, long long oh, long long os,
                         int dt16, hipStream_t st, bool one_side) {
    const FlashStrides sd{qh, qs, kh, ks, oh, os};
    if (dt16 == 0) {
        if (d == 128) return flash_launch<bf16, 128>((const bf16*)q, (const bf16*)k, (const bf16*)v, (bf16*)out, hq, hkv, q_len, kv_len, scale, sd, st, nullptr, nullptr, FlashWindow{}, FlashMany{}, one_side);
        return flash_launch<bf16, 64>((const bf16*)q, (const bf16*)k, (const bf16*)v, (bf16*)out, hq, hkv, q_len, kv_len, scale, sd, st, nullptr, nullptr, FlashWindow{}, FlashMany{}, one_side);
    }
    if (d == 128) return flash_launch<f16, 128>((const f16*)q, (const f16*)k, (const f16*)v, (f16*)out, hq, hkv, q_len, kv_len, scale, sd, st, nullptr, nullptr, FlashWindow{}, FlashMany{}, one_side);
    return flash_launch<f16, 64>((const f16*)q, (const f16*)k, (const f16*)v, (f16*)out, hq, hkv, q_len, kv_len, scale, sd, st, nullptr, nullptr, FlashWindow{}, FlashMany{}, one_side);
}

// sliding-window causal attention with an optional output gate and distance bias (bf16, head_dim 64 / 128, one key head per query head or
// a divisor, scale > 0): ops_latent.hip, engine_stack.hip
pgk_status flash_window(const void* q, const void* k, const void* v, void* out, int hq, int hkv, int q_len, int kv_len, int d, float scale,
                        int window, const OutGate& gate, const float* slopes, long long qh, long long qs, long long kh, long long ks, long long oh,
                        long long os, hipStream_t st) {
    PGK_REQUIRE((d == 64 || d == 128) && window >= 1 && scale > 0.f && kv_len >= q_len, "flash_window: d=%d window=%d q_len=%d kv_len=%d", d, window, q_len, kv_len);
    const FlashStrides sd{qh, qs, kh, ks, oh, os};
    const FlashWindow win{window, gate, slopes, 1.0f / scale};
    if (slopes && d == 128) return flash_launch<bf16, 128, true, true>((const bf16*)q, (const bf16*)k, (const bf16*)v, (bf16*)out, hq, hkv, q_len, kv_len, scale, sd, st, nullptr, nullptr, win);
    if (slopes) return flash_launch<bf16, 64, true, true>((const bf16*)q, (const bf16*)k, (const bf16*)v, (bf16*)out, hq, hkv, q_len, kv_len, scale, sd, st, nullptr, nullptr, win);
    if (d == 128) return flash_launch<bf16, 128, true>((const bf16*)q, (const bf16*)k, (const bf16*)v, (bf16*)out, hq, hkv, q_len, kv_len, scale, sd, st, nullptr, nullptr, win);
    return flash_launch<bf16, 64, true>((const bf16*)q, (const bf16*)k, (const bf16*)v, (bf16*)out, hq, hkv, q_len, kv_len, scale, sd, st, nullptr, nullptr, win);
}

// engine entry (fp8 x fp8 prefill, bf16, head_dim 128, q_len > 128): causal attention whose result leaves as the o_proj's fp8
// operand - codes [q_len][hq * 128] + scales [q_len][hq] - instead of bf16 rows (FlashSplit::q8)
pgk_status flash_prefill_q8(const void* q, const void* k, const void* v, uint8_t* q8, float* q8s, int hq, int hkv, int q_len, int kv_len,
                            float scale, long long qh, long long qs, long long kh, long long ks, hipStream_t st) {
    PGK_REQUIRE(q8 && q8s && q_len > 128, "flash_prefill_q8: needs output buffers and q_len > 128 (got %d)", q_len);
    const FlashStrides sd{qh, qs, kh, ks, 0, 0};
    return flash_launch<bf16, 128>((const bf16*)q, (const bf16*)k, (const bf16*)v, nullptr, hq, hkv, q_len, kv_len, scale, sd, st, q8, q8s, FlashWindow{}, FlashMany{}, true);
}

int flash_items(FlashItem* items, const int* lens, const int* starts, const int* slots, int n) {
    int at = 0;
    for (int i = 0, row0 = 0; i < n; row0 += lens[i++])
        for (int t = ceil_div(lens[i], FL_BQ) - 1; t >= 0; --t) items[at++] = FlashItem{row0, lens[i], starts[i] + lens[i], slots[i] << 16 | t};
    auto keys = [](const FlashItem& a) { return a.kv_len - a.q_len + std::min((a.slot_tile & 0xFFFF) * FL_BQ + FL_BQ, a.q_len); };
    std::stable_sort(items, items + at, [&](const FlashItem& a, const FlashItem& b) { return keys(a) > keys(b); });
    return at;
}
pgk_status flash_many(const void* q, const void* k, const void* v, void* out, const FlashItem* items, int n_items, int rows, int longest, long long slot_stride, int hq,
                      int hkv, int d, float scale, long long qh, long long qs, long long kh, long long ks, long long oh, long long os, hipStream_t st) {
    const FlashStrides sd{qh, qs, kh, ks, oh, os};
    const FlashMany many{items, n_items, rows, slot_stride};
    if (d == 128) return flash_launch<bf16, 128>((const bf16*)q, (const bf16*)k, (const bf16*)v, (bf16*)out, hq, hkv, rows, longest, scale, sd, st, nullptr, nullptr, FlashWindow{}, many);
    return flash_launch<bf16, 64>((const bf16*)q, (const bf16*)k, (const bf16*)v, (bf16*)out, hq, hkv, rows, longest, scale, sd, st, nullptr, nullptr, FlashWindow{}, many);
}

}  // namespace pgk
