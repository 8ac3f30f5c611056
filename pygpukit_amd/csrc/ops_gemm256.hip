// Large-tile MFMA GEMMs for gfx950 (prefill at S >= 256):  C[M,N] = A[M,K] . W[N,K]^T
//
//   bf16:  A, W bf16, fp32 accumulate, bf16 C or fp32 "+=" (the engine's residual stream)
//   fp8 :  A, W OCP e4m3 with 128-wide block scales (see ops_fp8_gemm.hip for the contract), same outputs
//
// Structure: 256 x 256 output tile per workgroup, 8 waves as 2 (M) x 4 (N), 128 x 64 per wave = 8 x 4 MFMA tiles of
// 16 x 16 held in 128 accumulator registers; K tiles of 128 BYTES per row (64 bf16 / 128 fp8).  Both operand
// tiles go global -> LDS by LDS-DMA (global_load_lds_dwordx4: no staging registers, no ds_write pass), 16 bytes
// per lane, one wave-instruction = 8 rows x 128 B written linearly; the bank swizzle is applied on the SOURCE
// address (lane p of a row fetches chunk p ^ (row & 7)) and again on the fragment reads, so the LDS image is the
// XOR-swizzled one without a scatter.  Two LDS buffers (128 KiB): the DMA of tile t+1 is issued before the MFMAs
// of tile t; one counted wait + one raw barrier per K tile.  All LDS lives in ONE dynamic array (a second
// __shared__ object makes hipcc wait vmcnt(0) before every fragment read).
// Workgroup ids are remapped so that the tiles an XCD works on form a compact patch of the output (shared A / W
// panels stay in that XCD's L2).
//
// The reference calls CUTLASS / cuBLASLt here (native/ops/matmul/matmul.cu:142-235); nothing of theirs is used.

#include "gemm_epilogues.hip.h"
#include "gemv_core.hip.h"
#include "moe.hip.h"
#include "pgk_internal.h"

#include <climits>

namespace pgk {

typedef __bf16 bf16x8_g __attribute__((ext_vector_type(8)));
typedef float f32x4_g __attribute__((ext_vector_type(4)));
typedef int i32x8_g __attribute__((ext_vector_type(8)));

constexpr int G2_BM = 256, G2_BN = 256, G2_THREADS = 512;
constexpr int G2_TILE = 256 * 128;   // bytes of one operand tile

// byte offset of 16-byte chunk c (0..7) of row r in a [rows][128 B] tile
__device__ __forceinline__ int g2_off(int r, int c) { return r * 128 + ((c ^ (r & 7)) << 4); }

// fp8 image swizzle (see gemm256_fp8_kernel): (r & 7) ^ (5 for rows 8-15 of every 16)
__device__ __forceinline__ int g2_sw8(int r) { return (r & 7) ^ ((r & 8) ? 5 : 0); }

// One LDS-DMA wave-instruction: 64 lanes x 16 bytes from per-lane global addresses to LDS [lds_addr, +1024).
// Written as inline asm on purpose: issued through __builtin_amdgcn_global_load_lds, hipcc (ROCm 7.2) puts an
// s_waitcnt vmcnt(0) in front of the next ds_read of the kernel - it cannot tell the buffer being filled from the
// buffer being read - and the prefetch is drained the moment it is issued.  The waits that order these DMAs
// before the fragment reads are the explicit vmcnt + barrier pairs in the kernels below.
__device__ __forceinline__ void g2_dma16(const void* src, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(lds_addr) : "memory", "m0");
}
// the same with a wave-uniform 64-bit base (SGPR pair) and a per-lane 32-bit byte offset
__device__ __forceinline__ void g2_dma16_so(const void* sbase, uint32_t voff, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase), "s"(lds_addr) : "memory", "m0");
}
__device__ __forceinline__ uint32_t g2_lds_addr(const char* p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)p;
}

// workgroup id -> output tile: ids are dealt round-robin to the 8 XCDs, so XCD x owns ids x, x+8, ...; give it a
// contiguous run of tiles, and walk the tiles in groups of 4 tile-rows so a run is a compact patch.
__device__ __forceinline__ void g2_tile_of(int id, int nwg, int ntm, int ntn, int& tm, int& tn) {
    const int q = nwg / 8, r = nwg % 8, xcd = id % 8, idx = id / 8;
    const int t = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + idx;   // bijective for any nwg
    constexpr int GM = 4;
    const int per_group = GM * ntn, g = t / per_group, first = g * GM;
    const int gsz = min(ntm - first, GM), in = t % per_group;
    tm = first + in % gsz;
    tn = in / gsz;
}

// ---- bf16 C tiles in LDS, for the epilogues.  Kernels with such a tile multiply W fragments by A fragments, so a lane of a 16 x 16 product holds four consecutive columns of
// one row (row lane & 15, columns 4 (lane >> 4) .. + 4) and puts them down in one 8-byte instruction, where four rows of a column took four of 2 bytes.
// 16-byte chunks are XOR-ed by the row so that the 16 rows of an instruction meet different banks; whole rows are read back.
//   us a launch, the other way and this: 1531 rows, K = 1024: SwiGLU (192 x 192) 23.5 / 23.0, QKV heads (192 x 128) 20.0 / 19.5; 256 x 192 tiles stored from registers, 4096
// rows, K = 4096, N = 6144 177 / 172.  Not for fp32 tiles (16 bytes for four of 4; += of N = 4096, K = 4096 107 / 113); and in the 256-row tiles that finish SwiGLU and
// heads where few of their rows are padding (gemm256_rows).
template <int ROWB> __device__ __forceinline__ int ct_off(int row, int byte) {
    static_assert(ROWB % 128 == 0, "chunks are exchanged in groups of 8, or of 16");
    const int sw = ROWB % 256 == 0 ? row & 15 : (row >> 1) & 7;
    return row * ROWB + (((byte >> 4) ^ sw) << 4) + (byte & 15);
}
__device__ __forceinline__ uint2 ct_bf16(const f32x4_g& v) { return make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])); }

// ---- SwiGLU epilogue (EPI 2 of the kernels below): W is the fused [2 I, K] gate / up weight, the workgroup's 256 B-tile rows are
// gate rows [128 tn, +128) followed by up rows [I + 128 tn, +128), so output tile tn holds act columns [128 tn, +128): waves
// wc 0 / 1 hold gate columns, wc 2 / 3 the matching up columns.  The accumulators go to LDS as the bf16 tile the plain kernel
// would have stored ([256][256] bf16 = the 128 KiB the operand stages occupied; 2-byte writes, the 32-byte run of a lane
// quarter XOR-ed by q so the four quarters of a wave hit different banks), then 16 consecutive lanes take one row's 128
// act columns, 8 each: act = bf16(silu(g) * u) from the bf16-ROUNDED g and u - the arithmetic of swiglu_rows_kernel
// (engine.hip) on the values the plain epilogue stores, so the result is bit-identical to GEMM + swiglu_rows_kernel - and
// store 16 bytes of bf16, or (QOUT) 8 e4m3 codes with the row's scale for this 128-column block (absmax / 448 over the 16
// lanes, quantize_fp8_rows' contract): exactly the fp8 x fp8 down projection's A operand.  Saves the [M][2 I] bf16 round
// trip through HBM (Llama-3-8B shape, S = 4096: 235 MB written + read back = ~75 us of a 1.4 ms layer) and a launch.
template <bool QOUT, int TN = 4, bool ROWS = false>   // ROWS: a lane holds columns of a row (ct_off), otherwise rows of a column; TN = n-fragments per wave column: 4 = 128 act columns per tile; 3 = 96 (bf16 output only)
__device__ __forceinline__ void g2_swiglu_epilogue(char* smem, const f32x4_g (&acc)[8][TN], int tid, int m0, int tn, int M, int I,
                                                   void* outv, float* out_scales) {
    static_assert(TN == 4 || !QOUT, "the e4m3 epilogue needs whole 128-column scale blocks");
    constexpr int WN = TN * 16, ACT = 2 * WN, ROWB = 4 * WN * 2, CH = ACT / 8;       // act columns per tile, bytes per LDS row, 8-column chunks per row
    const int lane = tid & 63, wid = tid >> 6, wr = wid >> 2, wc = wid & 3, q = lane >> 4, l15 = lane & 15;
    __builtin_amdgcn_s_barrier();                    // every wave is past its last operand read (DMAs retired by the caller)
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            if constexpr (ROWS) {
                *reinterpret_cast<uint2*>(smem + ct_off<ROWB>(wr * 128 + i * 16 + l15, (wc * WN + j * 16 + q * 4) * 2)) = ct_bf16(acc[i][j]);
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int row = wr * 128 + i * 16 + q * 4 + r, colb = (wc * WN + j * 16 + l15) * 2;
                    *reinterpret_cast<bf16*>(smem + row * ROWB + (colb ^ (q << 5))) = from_f<bf16>(acc[i][j][r]);   // (row >> 2) & 3 == q; the XOR stays inside a 128-byte group
                }
            }
        }
    auto at = [&](int row, int byte) { return smem + (ROWS ? ct_off<ROWB>(row, byte) : row * ROWB + (byte ^ (((row >> 2) & 3) << 5))); };
    __syncthreads();
#pragma unroll
    for (int it = 0; it < 256 * CH / G2_THREADS; ++it) {
        const int item = it * G2_THREADS + tid, row = item / CH, c = item % CH;
        Vec<bf16> g, u;
        g.raw = *reinterpret_cast<const uint4*>(at(row, c * 16));
        u.raw = *reinterpret_cast<const uint4*>(at(row, ACT * 2 + c * 16));
        float gf[8], uf[8];
        g.to_float(gf);
        u.to_float(uf);
#pragma unroll
        for (int e = 0; e < 8; ++e) gf[e] = gf[e] / (1.0f + __expf(-gf[e])) * uf[e];
        g.from_float(gf);
        const size_t grow = (size_t)m0 + row;
        if constexpr (QOUT) {
            g.to_float(gf);
            float amax = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) amax = fmaxf(amax, fabsf(gf[e]));
            amax = group16_max(amax);
            const float sc = amax > 0.f ? amax / 448.0f : 1.0f;
            uint2 o;
            o.x = pack_fp8x4(gf[0] / sc, gf[1] / sc, gf[2] / sc, gf[3] / sc);
            o.y = pack_fp8x4(gf[4] / sc, gf[5] / sc, gf[6] / sc, gf[7] / sc);
            if (grow < (size_t)M) {
                *reinterpret_cast<uint2*>(reinterpret_cast<uint8_t*>(outv) + grow * I + tn * ACT + c * 8) = o;
                if (c == 0) out_scales[grow * (I >> 7) + tn] = sc;
            }
        } else {
            if (grow < (size_t)M) g.store(reinterpret_cast<bf16*>(outv) + grow * I + tn * ACT + c * 8);
        }
    }
}

// ---- fp32 "+=" epilogue (EPI 1) through LDS: the residual stream is read and written as whole 512-byte row segments ---------
// The direct form - every lane adds its 128 accumulators to 128 separate words, 16 lanes per 64 contiguous bytes - cost
// ~30-40 us per launch at the Llama shapes (o_proj 161 us against 121 for the bf16-store kernel of the same product), all of
// it exposed: a one-wave grid has no second tile to hide an epilogue behind.  Here, per 64-column quarter of the tile: the
// residual words are requested first (8 float4 per lane), the owning wave column puts its accumulators into LDS ([256][64]
// fp32 over the operand stages, lane quarters XOR-ed apart), and every lane adds and stores 8 float4 (256-byte row segments).
__device__ __forceinline__ void g2_accum_epilogue(char* smem, const f32x4_g (&acc)[8][4], int tid, int m0, int n0, int M, int N, float* C) {
    const int lane = tid & 63, wid = tid >> 6, wr = wid >> 2, wc = wid & 3, q = lane >> 4, l15 = lane & 15;
    // one pass per 64-column quarter (= one wave column): 8 float4 per lane in flight (16 - halves - spilled in these kernels)
#pragma unroll 1
    for (int h = 0; h < 4; ++h) {
        float4 old[8];
#pragma unroll
        for (int it = 0; it < 8; ++it) {
            const int item = it * G2_THREADS + tid, row = item >> 4, c = item & 15;
            old[it] = *reinterpret_cast<const float4*>(C + (size_t)min(m0 + row, M - 1) * N + min(n0 + h * 64 + c * 4, N - 4));
        }
        __syncthreads();                             // operand stages (h = 0) / the previous quarter's tile are no longer read
        if (wc == h) {
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int row = wr * 128 + i * 16 + q * 4 + r, colb = (j * 16 + l15) * 4;
                        *reinterpret_cast<float*>(smem + row * 256 + (colb ^ (q << 6))) = acc[i][j][r];      // (row >> 2) & 3 == q
                    }
        }
        __syncthreads();
#pragma unroll
        for (int it = 0; it < 8; ++it) {
            const int item = it * G2_THREADS + tid, row = item >> 4, c = item & 15, sw = ((row >> 2) & 3) << 6;
            float4 v = *reinterpret_cast<const float4*>(smem + row * 256 + ((c * 16) ^ sw));
            const int grow = m0 + row, gcol = n0 + h * 64 + c * 4;
            if (grow >= M || gcol >= N) continue;
            v.x += old[it].x; v.y += old[it].y; v.z += old[it].z; v.w += old[it].w;
            *reinterpret_cast<float4*>(C + (size_t)grow * N + gcol) = v;
        }
    }
}

// ---- QKV-heads epilogue (EPI 3 of the fp8 kernel, 5 of the bf16 one): the accumulators go to LDS as the bf16 tile the plain kernel would have stored (the layout of
// g2_swiglu_epilogue), a tile = 256 token rows x two head slots, 16 consecutive lanes take one (row, head) and finish it
// (HeadRows: per-head RMSNorm, RoPE, q -> qkv buffer, k / v -> cache): bit-identical to GEMM + qknorm_rope_kvwrite_kernel.
template <bool ROWS = false>
__device__ __forceinline__ void g2_qkv_heads_epilogue(char* smem, const f32x4_g (&acc)[8][4], int tid, int m0, int tn, int M, int N, bf16* qkv,
                                                      const QkvHeadArgs& hd) {
    const int lane = tid & 63, wid = tid >> 6, wr = wid >> 2, wc = wid & 3, q = lane >> 4, l15 = lane & 15;
    const int c = tid & 15, r0 = tid >> 4;                   // 16 lanes take both heads of rows r0 + 32 i, whose angles they share
    HeadRows<8> hr;
    hr.places(m0 + r0, 32, M, hd);
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if constexpr (ROWS) {
                *reinterpret_cast<uint2*>(smem + ct_off<512>(wr * 128 + i * 16 + l15, (wc * 64 + j * 16 + q * 4) * 2)) = ct_bf16(acc[i][j]);
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int row = wr * 128 + i * 16 + q * 4 + r, colb = (wc * 64 + j * 16 + l15) * 2;
                    *reinterpret_cast<bf16*>(smem + row * 512 + (colb ^ (q << 5))) = from_f<bf16>(acc[i][j][r]);
                }
            }
        }
    hr.angles(c, 2 * tn, hd);
    __syncthreads();
#pragma unroll
    for (int h = 0; h < 2; ++h)
        hr.finish(c, 2 * tn + h, m0 + r0, 32, M, hd, qkv, N, [&](int i, float (&x)[8]) {
            const int row = i * 32 + r0, byte = h * 256 + c * 16;
            Vec<bf16> raw;
            raw.raw = *reinterpret_cast<const uint4*>(smem + (ROWS ? ct_off<512>(row, byte) : row * 512 + (byte ^ (((row >> 2) & 3) << 5))));
            raw.to_float(x);
        });
}

template <int EPI>   // 0: bf16 C store (+bias); 1: fp32 C +=
__global__ __launch_bounds__(G2_THREADS) void gemm256_bf16_kernel(const bf16* A, const bf16* W, const bf16* bias, void* Cv,
                                                                   int M, int N, int K, int ntm, int ntn) {
    extern __shared__ __attribute__((aligned(16))) char g2_smem[];   // A[2] | W[2]
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int wr = wid >> 2, wc = wid & 3, q = lane >> 4, l15 = lane & 15;
    int tm, tn;
    g2_tile_of(blockIdx.x, ntm * ntn, ntm, ntn, tm, tn);
    const int m0 = tm * G2_BM, n0 = tn * G2_BN;

    // DMA sources: wave w moves rows 32w .. 32w+31 of each tile, 8 rows per instruction; lane -> (row l>>3, chunk p = l&7)
    const int drow = wid * 32 + (lane >> 3);
    const int dchunk = (lane & 7) ^ (lane >> 3);            // logical chunk that lands at linear position l&7
    const bf16* a_src[4];
    const bf16* w_src[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        a_src[i] = A + (size_t)min(m0 + drow + 8 * i, M - 1) * K + dchunk * 8;
        w_src[i] = W + (size_t)min(n0 + drow + 8 * i, N - 1) * K + dchunk * 8;
    }
    const uint32_t lds0 = g2_lds_addr(g2_smem);
    auto stage = [&](int kt, int buf) {
        const uint32_t a_dst = __builtin_amdgcn_readfirstlane(lds0 + buf * G2_TILE + wid * 4096);
        const uint32_t w_dst = __builtin_amdgcn_readfirstlane(lds0 + (2 + buf) * G2_TILE + wid * 4096);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            g2_dma16(a_src[i] + (size_t)kt * 64, a_dst + i * 1024);
            g2_dma16(w_src[i] + (size_t)kt * 64, w_dst + i * 1024);
        }
    };

    f32x4_g acc[8][4];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_g{0.f, 0.f, 0.f, 0.f};

    // fragment read offsets: row = base + l15 (base a multiple of 16), chunk = ks*4 + q
    const int f_off0 = l15 * 128 + (((0 + q) ^ (l15 & 7)) << 4);
    const int f_off1 = l15 * 128 + (((4 + q) ^ (l15 & 7)) << 4);
    const int a_base = wr * 128 * 128, w_base = wc * 64 * 128;

    const int nk = K / 64;
    stage(0, 0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    for (int kt = 0; kt < nk; ++kt) {
        const int buf = kt & 1;
        if (kt + 1 < nk) stage(kt + 1, buf ^ 1);
        const char* As = g2_smem + buf * G2_TILE + a_base;
        const char* Ws = g2_smem + (2 + buf) * G2_TILE + w_base;
        // Both k-steps' fragments are requested before the first MFMA: the second set's LDS latency runs under the
        // first 32 MFMAs (one wave cannot rely on its SIMD neighbour for that).  The sched_barriers pin this order;
        // left alone, hipcc keeps only two reads in flight and waits for one before every group of 4 MFMAs.
        uint4 fa0[8], fb0[4], fa1[8], fb1[4];
#pragma unroll
        for (int i = 0; i < 8; ++i) fa0[i] = *reinterpret_cast<const uint4*>(As + i * 2048 + f_off0);
#pragma unroll
        for (int j = 0; j < 4; ++j) fb0[j] = *reinterpret_cast<const uint4*>(Ws + j * 2048 + f_off0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 8; ++i) fa1[i] = *reinterpret_cast<const uint4*>(As + i * 2048 + f_off1);
#pragma unroll
        for (int j = 0; j < 4; ++j) fb1[j] = *reinterpret_cast<const uint4*>(Ws + j * 2048 + f_off1);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_g, fa0[i]),
                                                                    __builtin_bit_cast(bf16x8_g, fb0[j]), acc[i][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_g, fa1[i]),
                                                                    __builtin_bit_cast(bf16x8_g, fb1[j]), acc[i][j], 0, 0, 0);
        __builtin_amdgcn_s_setprio(0);
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
    }

    // C/D map: col = lane & 15, row = (lane >> 4) * 4 + reg
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int col = n0 + wc * 64 + j * 16 + l15;
        if (col >= N) continue;
        float b = 0.f;
        if constexpr (EPI == 0) b = bias ? to_f(bias[col]) : 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = m0 + wr * 128 + i * 16 + q * 4 + r;
                if (row >= M) continue;
                if constexpr (EPI == 0) reinterpret_cast<bf16*>(Cv)[(size_t)row * N + col] = from_f<bf16>(acc[i][j][r] + b);
                else reinterpret_cast<float*>(Cv)[(size_t)row * N + col] += acc[i][j][r];
            }
    }
}

// ---- bf16, staggered phases: the two waves of a SIMD alternate between "read + DMA issue" and "32 MFMAs" ---------
// In the kernel above both waves of a SIMD leave each barrier together, request fragments together and want the MFMA
// pipe together: the pipe idles while both wait (57 % busy).  Here the stage is half a K tile ([256 rows][32 k] per
// operand, 16 KiB each; three in flight) and a wave's work on stage s is two phases,
//     A(s): request the 12 fragments of stage s, issue the DMA of stage s+3, wait for the fragments  | barrier
//     B(s): 32 MFMAs                                                                                  | barrier
// with waves 4-7 (the second wave of every SIMD) running ONE PHASE BEHIND waves 0-3 (one extra barrier up front, one
// at the end for the others): whenever one wave of a SIMD multiplies, the other one reads.  A stage is refilled one
// phase after its last reader finished (lgkmcnt(0) before that phase's barrier); its arrival is ordered by a counted
// vmcnt(8) - two younger stages may stay in flight - at the end of the phase before the first group reads it, which
// is B(s) for waves 0-3 and A(s) for waves 4-7.  DMAs past the end of K re-read the last stage (never consumed) so the
// count is constant.  64-byte rows: chunk c of row r at r*64 + ((c ^ ((r >> 2) & 2)) << 4).  ds_read_b128 is served in the
// lane groups {0-3, 12-15, 20-27}, {4-11, 16-19, 28-31} (+32), not in runs of 16 lanes: the first version's swizzle
// (r >> 2) & 3 was conflict-free for runs of 16 and 2-way conflicted for the real groups (SQ_LDS_BANK_CONFLICT = half of
// SQ_LDS_IDX_ACTIVE on the round-2 kernel); (r >> 2) & 2 is conflict-free for them (exhaustive check; counter 0 in
// profiles/r03_gemm256s_pmc.txt).
// What the loop waits for is not latency (eight stages in flight instead of three: the same time) but the rate at which the LDS-DMA delivers, and
// that depends on how a wave instruction's 1 KiB lies in memory.  L2-resident, all CUs: 33 TB/s for whole 128-byte lines, 31 for 64-byte halves in
// passing pairs, 9.7 for a fragment-major block fetched in another order than memory's.  So
//   * the packed W block goes to LDS as it lies, which is also the image a fragment read wants (lane l reads chunk l: no swizzle);
//   * A comes two stages at a time, 8 rows x 128 B per instruction, into a ring of G2S_ARING half-stage slots of its own: image [rows][128 B], chunk
//     c of row r at c ^ (r & 7) (g2_off), conflict-free in the groups above too.  A pair is requested at the even stages, 4 stages ahead, so between
//     any stage and its wait lie two W stages and one A pair: the counts of the three-in-flight scheme, vmcnt(8).
// M = 4096, packed W, us, both changes: N = 4096, K = 14336 396 -> 344; N = 14336 (SwiGLU), K = 4096 774 -> 704; N = 6144, K = 4096 198 -> 171.  Row-major
// W keeps its 64-byte rows (ring slots for pairs of both operands would not fit): 743 -> 719 for the SwiGLU product.
// TN = n-fragments per wave column: 4 = 256-column tiles; 3 = 192-column tiles (EPI 0 only), for shapes whose 256-tiles leave a
// half-empty last round: Llama's QKV (4096 x 6144) is 384 tiles = 1.5 rounds of the 256 CUs, 512 tiles of 256 x 192 are two
// full rounds of three quarters the work.  The W stage then has 192 rows = 12 DMA instructions: waves 0-3 move two (rows 0-127),
// waves 4-7 one (rows 128-191), so the "two younger stages in flight" count is vmcnt(8) for the former, vmcnt(6) for the latter.
constexpr int G2S_ARING = 6;      // slots of A, in stages
constexpr size_t G2S_LDS = (G2S_ARING + 4) * (size_t)256 * 64;
// EPI 0: bf16 C store (+bias); 1: fp32 C +=; 2: SwiGLU (W = fused gate / up rows, N = I act columns, C = bf16 act [M][I]); 3: xIELU, 4: gelu, bf16 store;
// 5: QKV heads (QkvHeadArgs; a tile holds two head slots, N % 256 == 0).  Qwen3-0.6B, 3365 rows: 38 us and 14 of the separate pass -> 38.
// EPI 0, 2, 5: rows scaled by NormIn where given.
template <int EPI, int TN = 4, bool ROWS = false>   // ROWS: a lane holds columns of a row (ct_off; gemm256_rows, gemm256_rows_store)
__global__ __launch_bounds__(G2_THREADS) void gemm256s_bf16_kernel(const bf16* A, const bf16* W, const bf16* bias, void* Cv,
                                                                    int M, int N, int K, int ntm, int ntn, int packed, ActArgs xa, QkvHeadArgs hd, NormIn ni) {
    static_assert(TN == 4 || (TN == 3 && EPI != 1 && EPI != 5), "192-column tiles: no +=, no heads");
    extern __shared__ __attribute__((aligned(16))) char g2_smem[];   // A: G2S_ARING slots of 16 KiB | W: 4 stages of 16 KiB
    constexpr int HALF = 256 * 64, BN = TN * 64, WN = TN * 16;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int wr = wid >> 2, wc = wid & 3, q = lane >> 4, l15 = lane & 15;
    const int late = __builtin_amdgcn_readfirstlane(wr);     // wave-uniform by construction: scalar branches around barriers
    int tm, tn;
    g2_tile_of(blockIdx.x, ntm * ntn, ntm, ntn, tm, tn);
    const int m0 = tm * G2_BM, n0 = tn * BN;

    const int drow = wid * 32 + (lane >> 2);                 // one DMA instruction of W = 16 rows x 64 B
    const int dchunk = (lane & 3) ^ ((lane >> 4) & 2);      // = (lane & 3) ^ g2s_sw(row & 15), row & 15 = lane >> 2
    const bf16* a_src[4];                                    // of A: 8 rows x 128 B, two stages
#pragma unroll
    for (int i = 0; i < 4; ++i) a_src[i] = A + (size_t)min(m0 + wid * 32 + 8 * i + (lane >> 3), M - 1) * K + ((lane & 7) ^ (lane >> 3)) * 8;
    // B-tile row r of an EPI-2 workgroup: gate row 128 tn + r for r < 128, up row N + 128 tn + (r - 128) after that (N = I)
    const int wtile_row = (TN == 4 || !late) ? drow : 128 + (wid - 4) * 16 + (lane >> 2);
    constexpr int GATE = TN * 32;     // EPI 2: gate rows per B tile (128 / 96), the matching up rows follow
    const int wrow = (EPI == 2) ? (wtile_row < GATE ? tn * GATE + wtile_row : N + tn * GATE + wtile_row - GATE) : n0 + wtile_row;
    const int wlast = (EPI == 2) ? 2 * N - 1 : N - 1;
    // W row-major [rows][K], or (packed) the fragment-major copy of ops_pkgemm.hip: block (16-row tile nt, k-step ks) = 1 KiB at
    // ((nt K/32 + ks) 64 + chunk 16 + row) 8 elements.  One DMA instruction moves 16 rows x 32 k = exactly one such block, as it lies,
    // and a stage advances 512 elements.
    const bf16 *w_src0, *w_src1;
    const int wk = packed ? 512 : 32;
    if (packed) {
        const int r_in = lane >> 2, nt_last = (wlast >> 4);
        w_src0 = W + ((size_t)min((wrow - r_in) >> 4, nt_last) * (K >> 5) * 64 + lane) * 8;
        w_src1 = W + ((size_t)min((wrow - r_in + 16) >> 4, nt_last) * (K >> 5) * 64 + lane) * 8;
    } else {
        w_src0 = W + (size_t)min(wrow, wlast) * K + dchunk * 8;
        w_src1 = W + (size_t)min(wrow + 16, wlast) * K + dchunk * 8;
    }
    const uint32_t lds0 = g2_lds_addr(g2_smem);
    const int nh = K / 32;
    // past the end of K the last stage is read again (never consumed): the counts below stay constant
    auto stage_a = [&](int h, int at) {                      // `at`: byte offset of the ring's slot
        const int k = min(h, nh - 2) * 32;
        const uint32_t a_dst = __builtin_amdgcn_readfirstlane(lds0 + at + wid * 4096);
#pragma unroll
        for (int i = 0; i < 4; ++i) g2_dma16(a_src[i] + k, a_dst + i * 1024);
    };
    auto stage_w = [&](int h, int buf) {
        const size_t kw = (size_t)min(h, nh - 1) * wk;
        const uint32_t w_dst = __builtin_amdgcn_readfirstlane(lds0 + (G2S_ARING + buf) * HALF + wid * 2048);
        if (TN == 4 || !late) {
            g2_dma16(w_src0 + kw, w_dst);
            g2_dma16(w_src1 + kw, w_dst + 1024);
        } else {
            g2_dma16(w_src0 + kw, __builtin_amdgcn_readfirstlane(lds0 + (G2S_ARING + buf) * HALF + 128 * 64 + (wid - 4) * 1024));
        }
    };
    // "this wave's share of the oldest of three stages in flight has landed"
    auto wait_two_younger = [&]() {
        if constexpr (TN == 4) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
        else if (late) asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    };

    f32x4_g acc[8][TN];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = f32x4_g{0.f, 0.f, 0.f, 0.f};
    const int w_off = packed ? lane * 16 : l15 * 64 + ((q ^ ((l15 >> 2) & 2)) << 4);
    const int a_off0 = l15 * 128 + ((q ^ (l15 & 7)) << 4), a_off1 = l15 * 128 + (((4 + q) ^ (l15 & 7)) << 4);
    const int a_base = wr * 128 * 128, w_base = G2S_ARING * HALF + wc * WN * 64;
    uint4 fa[8], fb[TN];

    stage_a(0, 0);
    stage_w(0, 0);
    stage_a(2, 2 * HALF);
    stage_w(1, 1);
    stage_w(2, 2);
    int a_cur = 0;                                           // ring slot of A's stage s
    // 1 / rms of row tid, where a register is left for it through the loop
    constexpr bool EARLY = (EPI == 0 || EPI == 2) && TN == 3;
    float mine = 0.f;
    if constexpr (EARLY) {
        if (ni.ss && tid < 256) mine = norm_in_scale(ni, min(m0 + tid, M - 1), M, K);
    }
    wait_two_younger();
    __builtin_amdgcn_s_barrier();
    if (late) __builtin_amdgcn_s_barrier();                  // waves 4-7 start one phase behind
#define G2S_STEP(S, BUF)                                                                                     \
    {   /* phase A */                                                                                        \
        const char* As = g2_smem + a_cur + a_base + (((BUF) & 1) ? a_off1 : a_off0);                           \
        const char* Ws = g2_smem + (BUF) * HALF + w_base + w_off;                                        \
        _Pragma("unroll") for (int i = 0; i < 8; ++i) fa[i] = *reinterpret_cast<const uint4*>(As + i * 2048); \
        _Pragma("unroll") for (int j = 0; j < TN; ++j) fb[j] = *reinterpret_cast<const uint4*>(Ws + j * 1024); \
        __builtin_amdgcn_sched_barrier(0);                                                                   \
        if (((BUF) & 1) == 0) {                                                                              \
            const int a_new = a_cur >= 2 * HALF ? a_cur - 2 * HALF : a_cur + 4 * HALF;                       \
            stage_a((S) + 4, a_new);                                                                         \
        }                                                                                                    \
        stage_w((S) + 3, ((BUF) + 3) & 3);                                                                   \
        if (((BUF) & 1) == 1) a_cur = a_cur == 4 * HALF ? 0 : a_cur + 2 * HALF;                              \
        if (late) wait_two_younger();                                                                        \
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                                                   \
        __builtin_amdgcn_s_barrier();                                                                        \
        __builtin_amdgcn_sched_barrier(0);                                                                   \
        /* phase B */                                                                                        \
        __builtin_amdgcn_s_setprio(1);                                                                       \
        _Pragma("unroll") for (int i = 0; i < 8; ++i)                                                        \
            _Pragma("unroll") for (int j = 0; j < TN; ++j)                                                   \
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_g, ROWS ? fb[j] : fa[i]),     \
                                                                    __builtin_bit_cast(bf16x8_g, ROWS ? fa[i] : fb[j]), acc[i][j], 0, 0, 0); \
        __builtin_amdgcn_s_setprio(0);                                                                       \
        __builtin_amdgcn_sched_barrier(0);                                                                   \
        if (!late) wait_two_younger();                                                                       \
        __builtin_amdgcn_s_barrier();                                                                        \
    }
    int s = 0;
    for (; s + 4 <= nh; s += 4) {
        G2S_STEP(s, 0) G2S_STEP(s + 1, 1) G2S_STEP(s + 2, 2) G2S_STEP(s + 3, 3)
    }
    if (s < nh) {   // K % 64 == 0: an even number of stages, so two remain at most
        G2S_STEP(s, 0) G2S_STEP(s + 1, 1)
    }
#undef G2S_STEP
    if (!late) __builtin_amdgcn_s_barrier();                 // match the extra barrier of waves 4-7
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");         // retire the phantom DMAs before the LDS is given back

    if constexpr (EPI == 0 || EPI == 2 || EPI == 5) {
        if (ni.ss) {
            float* inv = reinterpret_cast<float*>(g2_smem + 256 * 512);          // behind the epilogues' tile
            if (!EARLY && tid < 256) mine = norm_in_scale(ni, min(m0 + tid, M - 1), M, K);
            __builtin_amdgcn_s_barrier();                    // every wave is past its last operand read
            if (tid < 256) inv[tid] = mine;
            __syncthreads();
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                f32x4_g f;
                if constexpr (ROWS) {
                    const float one = inv[wr * 128 + i * 16 + l15];
                    f = f32x4_g{one, one, one, one};
                } else f = *reinterpret_cast<const f32x4_g*>(inv + wr * 128 + i * 16 + q * 4);
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[i][j] *= f;
            }
        }
    }
    if constexpr (EPI == 2) {
        g2_swiglu_epilogue<false, TN, ROWS>(g2_smem, acc, tid, m0, tn, M, N, Cv, nullptr);
        return;
    }
    if constexpr (EPI == 5) {
        g2_qkv_heads_epilogue<ROWS>(g2_smem, acc, tid, m0, tn, M, N, reinterpret_cast<bf16*>(Cv), hd);
        return;
    }
    if constexpr (EPI == 1 && TN == 4) {
        if ((N & 3) == 0) {       // whole float4s per row (every engine shape); otherwise the word-wise form below
            g2_accum_epilogue(g2_smem, acc, tid, m0, n0, M, N, reinterpret_cast<float*>(Cv));
            return;
        }
    }
    if constexpr (!ROWS) {                                   // EPI 1: N % 4 != 0
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int col = n0 + wc * WN + j * 16 + l15;
            if (col >= N) continue;
            float b = 0.f;
            if constexpr (EPI == 0) b = bias ? to_f(bias[col]) : 0.f;
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int row = m0 + wr * 128 + i * 16 + q * 4 + r;
                    if (row >= M) continue;
                    if constexpr (EPI == 0) reinterpret_cast<bf16*>(Cv)[(size_t)row * N + col] = from_f<bf16>(acc[i][j][r] + b);
                    else if constexpr (EPI == 3) reinterpret_cast<bf16*>(Cv)[(size_t)row * N + col] = from_f<bf16>(xielu<false>(acc[i][j][r], xa.pos, xa.neg));
                    else if constexpr (EPI == 4) reinterpret_cast<bf16*>(Cv)[(size_t)row * N + col] = from_f<bf16>(gelu_erf(acc[i][j][r]));
                    else reinterpret_cast<float*>(Cv)[(size_t)row * N + col] += acc[i][j][r];
                }
        }
        return;
    }
    // four columns of a row to a lane: one 8-byte store (gemm256_rows_store: every row is aligned to it)
    bf16* C = reinterpret_cast<bf16*>(Cv);
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int col = n0 + wc * WN + j * 16 + q * 4;
        if (col >= N) continue;
        float b[4] = {0.f, 0.f, 0.f, 0.f};
        if constexpr (EPI == 0) {
            if (bias) {
#pragma unroll
                for (int r = 0; r < 4; ++r) b[r] = to_f(bias[col + r]);
            }
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int row = m0 + wr * 128 + i * 16 + l15;
            if (row >= M) continue;
            f32x4_g v = acc[i][j];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if constexpr (EPI == 0) v[r] += b[r];
                else if constexpr (EPI == 3) v[r] = xielu<false>(v[r], xa.pos, xa.neg);
                else if constexpr (EPI == 4) v[r] = gelu_erf(v[r]);
            }
            *reinterpret_cast<uint2*>(C + (size_t)row * N + col) = ct_bf16(v);
        }
    }
}

// ---- bf16, smaller tiles: four waves multiply, four others fetch ------------------------------------------------------------
// For the shapes too small for 192 tiles of 256 x 256.  Tiles of 32 WM x 32 WN, 2 x 2 waves of 16 WM x 16 WN, stages of 32 k in the images, rings and
// counts of gemm256s (A a pair of stages at a time in whole lines, packed W as it lies).  A wave that issues an LDS-DMA instruction stands still until
// the CU's one texture path has taken its 64 addresses, 20 clocks and those of the waves in front of it: with the DMA in the multiplying waves a stage
// of a 128 x 128 tile took 0.25 us with one workgroup on the CU, half of it DMA issue (0.19 without the fragment reads, 0.12 for the DMA alone, 0.11 for
// the products alone).  So waves 4-7 issue all of it and waves 0-3 never do; the fragments of stage s + 1 are requested between the products of stage s,
// each into the registers its row of products has just read (W's, and the last row's, into a second set).  0.17-0.18 us a stage.
// One barrier per stage: behind it stage s + 1 has landed (the DMA waves have waited for their shares) and stage s has been read, so W of s + RW and,
// where s is odd, A of s + RA - 1 and s + RA take its place.
//   us a launch, before / after (K = 1024, packed W): 1531 rows, N = 6144 28.0 / 23.0 on 192 x 192 tiles, N = 4096 20.3 / 16.6 on 192 x 128; 384 rows,
//   N = 6144 12.7 / 10.8; K = 3072, N = 1024, 3365 rows 28.3 / 23.4.
// blockIdx.y = K split (EPI 2: fp32 slab z of [splits][M][N], summed by the consumer).
// Epilogue through LDS, by all eight waves: the tile as fp32 (as bf16 where the values are rounded to it first anyway, EPI 3 and 4) with the lane
// quarters XOR-ed apart, then back as rows for coalesced stores (EPI 1: float4 read-modify-write of the residual stream, all loads issued before the first
// store).
// EPI 0: bf16 C store (+bias); 1: fp32 C +=; 2: fp32 split-K slab; 3: QKV heads (QkvHeadArgs: tile column = head slot);
// 4: SwiGLU (W = fused gate / up rows, N = I act columns, C = bf16 act [M][I]; tile tn = act columns [16 WN tn, +16 WN)); 5: xIELU, 7: gelu, bf16 store;
// 8: 1, and what the next RMSNorm leaves to do (NormOut); 9: fp32 store and each row's best column of the tile (BestOut).  EPI 0, 3, 4: rows scaled by NormIn where given
// GRP: rows sorted by expert (GroupArgs), every tile with its expert's weight; EPI 4, 7, or 6: bf16 rows times their weight, each at its place
constexpr int GP_THREADS = 512;
// stages of W that the ring holds; A's has two more.  The smaller tiles' stages are shorter, and latency asks for more of them
constexpr int gemmp_ring(int WM, int WN) { return WM * WN >= 16 || (WM == 2 && WN == 4) ? 4 : 6; }
// Small tiles, whose stages are over before a barrier and the reads behind it are (gemmp_kg): the waves split K as well.  Of a pair of stages one wave of two multiplies the
// first, its partner the second, each for a piece of 32 WM x 16 WN; one barrier a pair, fewer fragment reads, and the partners trade halves of their sums at the end.  What is left is
// the rate of the LDS-DMA, 85 to 110 bytes a ns and CU.  Us a launch, the 2 x 2 split / this: K = 2048, N = 1024: 1531 rows, 96 x 64 13.0 / 12.1, 1000 rows, 64 x 64 10.4 / 9.1; K = 3072
// 17.5 / 16.3 and 13.6 / 12.1.  Only in front of the residual epilogue: SwiGLU's on 64 x 64 (K = 1024, N = 6144, 93 rows) took 5.9 / 5.3 alone, but 0.989 and 0.998 times the speed in a prompt of 93 and a step of
// 64 sequences.  (64 x 128 has no registers for it: twice the time.)
constexpr bool gemmp_kg(int EPI, int WM, int WN) { return WM == 1 || (EPI == 8 && WN == 2 && WM <= 3); }
constexpr int gemmp_pairs(int WM, int WN) { return WM == 1 ? 6 : WM == 2 ? 5 : 4; }      // pairs of stages in that ring: at most 80 KiB, two workgroups a CU
template <int EPI, int WM, int WN> constexpr size_t gemmp_lds() {
    constexpr bool B16 = EPI == 3 || EPI == 4;
    const size_t RW = gemmp_ring(WM, WN), tile = (size_t)(32 * WM) * (32 * WN) * (B16 ? 2 : 4);
    const size_t ring = gemmp_kg(EPI, WM, WN) ? gemmp_pairs(WM, WN) * (size_t)(32 * (WM + WN) * 128) : (RW + 2) * (size_t)(32 * WM * 64) + RW * (size_t)(32 * WN * 64);
    const size_t least = gemmp_kg(EPI, WM, WN) ? tile + 1024 + WM * WN * 4096 : tile;
    return ring > least ? ring : least;
}
struct BestOut { float* val; int* idx; };                    // [M][tiles of columns]
// s_waitcnt's counts are immediates, so the ends of the rings, where a step less is in flight each time, are unrolled over T = 0, 1, ...
template <int N> __device__ __forceinline__ void gp_wait() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
template <class F, int... T> __device__ __forceinline__ void gp_steps(std::integer_sequence<int, T...>, F f) { (f(std::integral_constant<int, T>{}), ...); }
template <int EPI, bool GRP, int WM, int WN>
__device__ __forceinline__ void gemmp_body(const bf16* A, const bf16* W, const bf16* bias, void* Cv,
                                           int M, int N, int K, int ntm, int ntn, int kps, const QkvHeadArgs& hd, int packed, const ActArgs& xa, const GroupArgs& ga, const NormIn& ni, const NormOut& no, const BestOut& bo) {
    extern __shared__ __attribute__((aligned(16))) char g2_smem[];   // A: RA slots of AH bytes | W: RW stages of WH
    constexpr int BM = 32 * WM, BN = 32 * WN, RW = gemmp_ring(WM, WN), RA = RW + 2, AH = BM * 64, WH = BN * 64, NA = WM, NW = WN / 2;   // NA, NW: DMA instructions of a wave for a pair of A's / a stage of W's
    constexpr bool KG = gemmp_kg(EPI, WM, WN);
    constexpr int GP_PAIRS = gemmp_pairs(WM, WN);
    constexpr bool B16 = EPI == 3 || EPI == 4, ROWS = B16, SCALED = !GRP && (EPI == 0 || EPI == 3 || EPI == 4), PARTS = SCALED && EPI == 4 && BM == 64;   // PARTS: may come as ni.ld says
    static_assert(!SCALED || BM <= 256, "a row for each of the waves that multiply");
    static_assert(WN % 2 == 0 && (EPI != 3 || WN == 4), "W's pieces divide by four waves; a head is 128 columns");
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    int tm, tn, m0;
    if constexpr (GRP) {
        ntm = *ga.n_tiles;
        if ((int)blockIdx.x >= ntm * ntn) return;            // (the grid is sized for the worst distribution)
    }
    g2_tile_of(blockIdx.x, ntm * ntn, ntm, ntn, tm, tn);
    if constexpr (GRP) {
        const MoeTile t = ga.tiles[tm];
        m0 = t.row0;
        M = t.row0 + t.rows;
        W += t.expert * ga.w_stride;
    } else m0 = tm * BM;
    const int n0 = tn * BN;
    const int kbeg = (int)blockIdx.y * kps, kend = min(K, kbeg + kps);
    const int nh = (kend - kbeg) / 32;                       // (kend - kbeg) % 64 == 0: an even number of stages

    f32x4_g acc[WM][WN];
    float mine = 0.f;                                        // 1 / rms of row tid (ni.ld: of tid / 4)
    const int part = (wid >> 1) & 1, kg = wid & 1;           // KG: which columns, which stage of a pair; behind the trade rows 16 WM kg .. of those columns
    const int wr = KG ? kg : part, wc = KG ? part : kg, q = lane >> 4, l15 = lane & 15;
    // EPI 1, 8: this thread's words of the residual stream, requested behind the last DMA and the last product
    constexpr int OLD = EPI == 1 || EPI == 8 ? BM * (BN / 4) / GP_THREADS : 0;
    float4 old[OLD > 0 ? OLD : 1];
    auto residual = [&]() {
#pragma unroll
        for (int it = 0; it < OLD; ++it)
            old[it] = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(Cv) + (size_t)min(m0 + (it * GP_THREADS + tid) / (BN / 4), M - 1) * N + min(n0 + tid % (BN / 4) * 4, N - 4));
    };
    if (wid >= 4) {
        const int pw = __builtin_amdgcn_readfirstlane(wid & 3);
        auto a_row = [&](int r) -> int {
            r = min(r, M - 1);
            if constexpr (GRP) return ga.div > 0 ? ga.order[r] / ga.div : r;
            else return r;
        };
        const bf16* a_src[NA];                               // 8 rows x 128 B, two stages
#pragma unroll
        for (int i = 0; i < NA; ++i) a_src[i] = A + (size_t)a_row(m0 + (pw * NA + i) * 8 + (lane >> 3)) * K + kbeg + ((lane & 7) ^ (lane >> 3)) * 8;
        // one instruction of W = 16 rows x 64 B of the row-major weight, or (packed) a block of the fragment-major copy as it lies: see gemm256s_bf16_kernel.
        // EPI 4: the tile's first half are gate rows, the second the matching up rows N further on (N = I)
        const bf16* w_src[NW];
        const int wk = packed ? 512 : 32, wlast = (EPI == 4) ? 2 * N - 1 : N - 1;
#pragma unroll
        for (int i = 0; i < NW; ++i) {
            const int r0 = (pw * NW + i) * 16;
            const int row = (EPI == 4) ? (r0 < BN / 2 ? tn * (BN / 2) + r0 : N + tn * (BN / 2) + r0 - BN / 2) : n0 + r0;
            if (packed) w_src[i] = W + (((size_t)min(row >> 4, wlast >> 4) * (K >> 5) + (kbeg >> 5)) * 64 + lane) * 8;
            else w_src[i] = W + (size_t)min(row + (lane >> 2), wlast) * K + kbeg + ((lane & 3) ^ ((lane >> 4) & 2)) * 8;
        }
        const uint32_t lds0 = g2_lds_addr(g2_smem);
        // a product of few stages fills the ring with its last one (never consumed)
        auto stage_a = [&](int h, int at) {                  // `at`: byte offset of the ring's slot
            const int k = min(h, nh - 2) * 32;
            const uint32_t dst = __builtin_amdgcn_readfirstlane(lds0 + at + pw * NA * 1024);
#pragma unroll
            for (int i = 0; i < NA; ++i) g2_dma16(a_src[i] + k, dst + i * 1024);
        };
        auto stage_w = [&](int h, int buf) {
            const size_t kw = (size_t)min(h, nh - 1) * wk;
            const uint32_t dst = __builtin_amdgcn_readfirstlane(lds0 + RA * AH + buf * WH + pw * NW * 1024);
#pragma unroll
            for (int i = 0; i < NW; ++i) g2_dma16(w_src[i] + kw, dst + i * 1024);
        };
        if constexpr (KG) {
            constexpr int PB = 2 * (AH + WH), EACH = NA + 2 * NW;     // bytes and DMA instructions of a pair
            auto stage_pair = [&](int p, int at) {
                const int h = min(2 * p, nh - 2);
                const uint32_t dst = __builtin_amdgcn_readfirstlane(lds0 + at);
#pragma unroll
                for (int i = 0; i < NA; ++i) g2_dma16(a_src[i] + h * 32, dst + (pw * NA + i) * 1024);
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int i = 0; i < NW; ++i) g2_dma16(w_src[i] + (size_t)(h + t) * wk, dst + 2 * AH + t * WH + (pw * NW + i) * 1024);
            };
#pragma unroll
            for (int p = 0; p < GP_PAIRS; ++p) stage_pair(p, p * PB);
            gp_wait<(GP_PAIRS - 1) * EACH>();                // pair 0
            __builtin_amdgcn_s_barrier();
            const int np = nh / 2;
            int at = 0, p = 0;
            for (; p + GP_PAIRS < np; ++p) {
                gp_wait<(GP_PAIRS - 2) * EACH>();            // pair p + 1; pair p is in registers behind the barrier
                __builtin_amdgcn_s_barrier();
                stage_pair(p + GP_PAIRS, at);
                at = at == (GP_PAIRS - 1) * PB ? 0 : at + PB;
            }
            residual();
            if (np >= GP_PAIRS) {
                gp_steps(std::make_integer_sequence<int, GP_PAIRS>{}, [&](auto t) {
                    constexpr int LEFT = GP_PAIRS - 2 - decltype(t)::value;
                    if constexpr (LEFT >= 0) gp_wait<LEFT * EACH + OLD>();
                    __builtin_amdgcn_s_barrier();
                });
            } else {
                gp_wait<OLD>();
                for (; p < np; ++p) __builtin_amdgcn_s_barrier();
            }
            __builtin_amdgcn_s_barrier();                    // the ring becomes the C tile
            __builtin_amdgcn_s_barrier();                    // the partners' trade
        } else {
        // between W of a stage and the wait for it: W of RW - 2 stages and their A
        constexpr int YOUNGER = (RW - 2) * NW + (RW - 2) / 2 * NA;
        stage_a(0, 0);
#pragma unroll
        for (int t = 0; t < RW; ++t) {
            if (t & 1) stage_a(t + 1, (t + 1) * AH);
            stage_w(t, t);
        }
        gp_wait<(RW - 1) * NW + RW / 2 * NA>();              // stage 0
        __builtin_amdgcn_s_barrier();
        if (nh >= RW + 2) {
            int at = 0, buf = 0, s = 0;
            for (; s + RW + 2 < nh; s += 2) {
                gp_wait<YOUNGER>();                          // stage s + 1
                __builtin_amdgcn_s_barrier();
                stage_w(s + RW, buf);
                gp_wait<YOUNGER>();
                __builtin_amdgcn_s_barrier();
                stage_a(s + RA, at);
                stage_w(s + RW + 1, buf + 1);
                at = at == (RA - 2) * AH ? 0 : at + 2 * AH;
                buf = buf == RW - 2 ? 0 : buf + 2;
            }
            gp_wait<YOUNGER>();
            __builtin_amdgcn_s_barrier();
            stage_w(s + RW, buf);
            gp_wait<YOUNGER>();
            __builtin_amdgcn_s_barrier();
            stage_w(s + RW + 1, buf + 1);
            residual();
            // the last RW stages: nothing is left to request.  (Requests for the last stage once more, which kept the counts constant, were waited for at the end.)
            gp_steps(std::make_integer_sequence<int, RW>{}, [&](auto t) {
                constexpr int LEFT = RW - 2 - decltype(t)::value, PAIRS = LEFT > 0 ? (LEFT + 1) / 2 - 1 : 0;      // stages requested behind the one waited for; their A
                if constexpr (LEFT >= 0) gp_wait<LEFT * NW + PAIRS * NA + OLD>();
                __builtin_amdgcn_s_barrier();
            });
        } else {
            residual();
            gp_wait<OLD>();
            for (int s = 0; s < nh; ++s) __builtin_amdgcn_s_barrier();
        }
        __builtin_amdgcn_s_barrier();                        // the stages become the C tile
        }
    } else {
        if constexpr (PARTS) {
            if (ni.ss && ni.ld) {                            // four threads to a row, 16 parts each
                const float* p = ni.ss + (size_t)min(m0 + (tid >> 2), M - 1) * 64 + (tid & 3) * 16;
                float4 v[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] = *reinterpret_cast<const float4*>(p + 4 * j);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int i = (tid & 3) * 16 + 4 * j;
                    mine += ((i < ni.n ? v[j].x : 0.f) + (i + 1 < ni.n ? v[j].y : 0.f)) + ((i + 2 < ni.n ? v[j].z : 0.f) + (i + 3 < ni.n ? v[j].w : 0.f));
                }
                mine += dpp_f<DPP_XOR1>(mine);
                mine += dpp_f<DPP_XOR2>(mine);
                mine = 1.0f / sqrtf(mine / K + ni.eps);
            }
        }
        if constexpr (SCALED && EPI != 0) {
            if (ni.ss && !(PARTS && ni.ld) && tid < BM) mine = norm_in_scale(ni, min(m0 + tid, M - 1), M, K);
        }
        const int w_off = packed ? lane * 16 : l15 * 64 + ((q ^ ((l15 >> 2) & 2)) << 4);
        const int a_off0 = l15 * 128 + ((q ^ (l15 & 7)) << 4), a_off1 = l15 * 128 + (((4 + q) ^ (l15 & 7)) << 4);
        auto frag = [&](const char* p) { return *reinterpret_cast<const bf16x8_g*>(p); };
        if constexpr (KG) {
            constexpr int FM = 2 * WM, PB = 2 * (AH + WH);
            f32x4_g big[FM][WN];
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < WN; ++j) big[i][j] = f32x4_g{0.f, 0.f, 0.f, 0.f};
            const char *a_at = g2_smem + (kg ? a_off1 : a_off0), *w_at = g2_smem + 2 * AH + kg * WH + part * 16 * WN * 64 + w_off;
            bf16x8_g fa[2][FM], fb[2][WN];
            auto fetch = [&](bf16x8_g (&A_)[FM], bf16x8_g (&W_)[WN], int at) {
#pragma unroll
                for (int i = 0; i < FM; ++i) A_[i] = frag(a_at + at + i * 2048);
#pragma unroll
                for (int j = 0; j < WN; ++j) W_[j] = frag(w_at + at + j * 1024);
            };
            int at = 0;                                      // ring slot of pair p
            auto step = [&](bf16x8_g (&A_)[FM], bf16x8_g (&W_)[WN], bf16x8_g (&nA)[FM], bf16x8_g (&nW)[WN]) {
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");    // pair p in registers: its place may be refilled
                __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_sched_barrier(0);
                at = at == (GP_PAIRS - 1) * PB ? 0 : at + PB;
                fetch(nA, nW, at);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int j = 0; j < WN; ++j) big[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ROWS ? W_[j] : A_[i], ROWS ? A_[i] : W_[j], big[i][j], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            };
            __builtin_amdgcn_s_barrier();
            fetch(fa[0], fb[0], 0);
            int s = 0;
            for (; s + 4 <= nh; s += 4) {
                step(fa[0], fb[0], fa[1], fb[1]);
                step(fa[1], fb[1], fa[0], fb[0]);
            }
            if (s < nh) step(fa[0], fb[0], fa[1], fb[1]);
            residual();
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");        // the reads past the last pair
            __builtin_amdgcn_s_barrier();
            // the lower rows of the piece to kg = 1, the upper ones to kg = 0; behind the C tile, which a faster wave may be writing
            char* trade = g2_smem + BM * BN * (B16 ? 2 : 4) + 1024 + lane * 16;
            auto hand = [&](int f, const f32x4_g& v) { *reinterpret_cast<f32x4_g*>(trade + ((wid ^ 1) * WM * WN + f) * 1024) = v; };
#pragma unroll
            for (int i = 0; i < WM; ++i)
#pragma unroll
                for (int j = 0; j < WN; ++j) {
                    if (kg == 0) { hand(i * WN + j, big[WM + i][j]); acc[i][j] = big[i][j]; }
                    else { hand(i * WN + j, big[i][j]); acc[i][j] = big[WM + i][j]; }
                }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
#pragma unroll
            for (int i = 0; i < WM; ++i)
#pragma unroll
                for (int j = 0; j < WN; ++j) acc[i][j] += *reinterpret_cast<const f32x4_g*>(trade + (wid * WM * WN + i * WN + j) * 1024);
        } else {
#pragma unroll
        for (int i = 0; i < WM; ++i)
#pragma unroll
            for (int j = 0; j < WN; ++j) acc[i][j] = f32x4_g{0.f, 0.f, 0.f, 0.f};
        const int a_base = wr * 16 * WM * 128, w_base = RA * AH + wc * 16 * WN * 64 + w_off;
        bf16x8_g fa[WM - 1], fl[2], fb[2][WN];               // A's rows but the last, the last, W's
        __builtin_amdgcn_s_barrier();
        {
            const char *As = g2_smem + a_base + a_off0, *Ws = g2_smem + w_base;
#pragma unroll
            for (int i = 0; i < WM - 1; ++i) fa[i] = frag(As + i * 2048);
            fl[0] = frag(As + (WM - 1) * 2048);
#pragma unroll
            for (int j = 0; j < WN; ++j) fb[0][j] = frag(Ws + j * 1024);
        }
        int a_cur = 0, w_cur = 0;                            // ring slots of stage s
#define GP_MFMA(I, F, P)                                                                                     \
    _Pragma("unroll") for (int j = 0; j < WN; ++j) acc[I][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ROWS ? fb[P][j] : F, ROWS ? F : fb[P][j], acc[I][j], 0, 0, 0); \
    __builtin_amdgcn_sched_barrier(0);
#define GP_STEP(BUF)                                                                                         \
    {                                                                                                        \
        constexpr int P = (BUF) & 1;                                                                         \
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   /* stage s in registers: its place may be refilled */ \
        __builtin_amdgcn_s_barrier();                                                                        \
        __builtin_amdgcn_sched_barrier(0);                                                                   \
        const int a_nxt = P ? (a_cur == (RA - 2) * AH ? 0 : a_cur + 2 * AH) : a_cur;                         \
        if constexpr (RW == 4) w_cur = (((BUF) + 1) & 3) * WH;                                               \
        else w_cur = w_cur == (RW - 1) * WH ? 0 : w_cur + WH;                                                \
        const char* As = g2_smem + a_nxt + a_base + (P ? a_off0 : a_off1);                                   \
        const char* Ws = g2_smem + w_cur + w_base;                                                           \
        _Pragma("unroll") for (int i = 0; i < WM - 1; ++i) {                                                 \
            GP_MFMA(i, fa[i], P)                                                                             \
            fa[i] = frag(As + i * 2048);                                                                     \
            if (i == 0) fl[P ^ 1] = frag(As + (WM - 1) * 2048);                                              \
            if (i < 2) {                                                                                     \
                _Pragma("unroll") for (int j = i * (WN / 2); j < (WM == 2 ? WN : (i + 1) * (WN / 2)); ++j) fb[P ^ 1][j] = frag(Ws + j * 1024); \
            }                                                                                                \
            __builtin_amdgcn_sched_barrier(0);                                                               \
        }                                                                                                    \
        GP_MFMA(WM - 1, fl[P], P)                                                                            \
        a_cur = a_nxt;                                                                                       \
    }
        int s = 0;
        for (; s + 4 <= nh; s += 4) {
            GP_STEP(0) GP_STEP(1) GP_STEP(2) GP_STEP(3)
        }
        if (s < nh) {
            GP_STEP(0) GP_STEP(1)
        }
#undef GP_STEP
#undef GP_MFMA
        residual();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the reads past the last stage, before the stages become the C tile
        __builtin_amdgcn_s_barrier();
        }
    }

    // rows of the tile: bf16 (ROWS: ct_off), or fp32, 64-byte group g at g ^ ((R >> 2) & 3), which is q for a lane's rows
    constexpr int ROWB = BN * (B16 ? 2 : 4);
    HeadRows<EPI == 3 ? BM / 32 : 1> hr;
    const int hrow = tid >> 4;                               // EPI 3: 16 consecutive lanes = one (token row, head)
    if constexpr (EPI == 3) hr.places(m0 + hrow, 32, M, hd);
    if constexpr (SCALED) {
        if (ni.ss) {
            float* inv = reinterpret_cast<float*>(g2_smem + BM * ROWB);          // behind the tile, where the last stages were
            if constexpr (EPI == 0) {                        // (held through the loop it is spilled; QKV of heads that are not 128 columns, and all where PGK_FUSED_EPILOGUES is 0)
                if (tid < BM) mine = norm_in_scale(ni, min(m0 + tid, M - 1), M, K);
            }
            if (PARTS && ni.ld) { if (tid < 256 && (tid & 3) == 0) inv[tid >> 2] = mine; }
            else if (tid < BM) inv[tid] = mine;
            __syncthreads();
            if (wid < 4) {
#pragma unroll
                for (int i = 0; i < WM; ++i) {
                    f32x4_g f;
                    if constexpr (ROWS) {
                        const float one = inv[wr * 16 * WM + i * 16 + l15];
                        f = f32x4_g{one, one, one, one};
                    } else f = *reinterpret_cast<const f32x4_g*>(inv + wr * 16 * WM + i * 16 + q * 4);
#pragma unroll
                    for (int j = 0; j < WN; ++j) acc[i][j] *= f;
                }
            }
        }
    }
    if (wid < 4) {
#pragma unroll
        for (int i = 0; i < WM; ++i)
#pragma unroll
            for (int j = 0; j < WN; ++j) {
                if constexpr (ROWS) {
                    *reinterpret_cast<uint2*>(g2_smem + ct_off<ROWB>(wr * 16 * WM + i * 16 + l15, (wc * 16 * WN + j * 16 + q * 4) * 2)) = ct_bf16(acc[i][j]);
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        *reinterpret_cast<float*>(g2_smem + (wr * 16 * WM + i * 16 + q * 4 + r) * ROWB + (((wc * 16 * WN + j * 16 + l15) * 4) ^ (q << 6))) = acc[i][j][r];
                }
            }
    }
    if constexpr (EPI == 3) hr.angles((tid & 15), tn, hd);
    auto tile4 = [&](int row, int byte) { return *reinterpret_cast<const float4*>(g2_smem + row * ROWB + (byte ^ (((row >> 2) & 3) << 6))); };
    if constexpr (EPI == 1 || EPI == 8) {
        const int c = tid % (BN / 4), gcol = n0 + c * 4;     // a thread's columns are the same in all its rows
        uint2 gamma = make_uint2(0, 0);
        if constexpr (EPI == 8) gamma = *reinterpret_cast<const uint2*>(no.gamma + min(gcol, N - 4));
        __syncthreads();
#pragma unroll
        for (int it = 0; it < OLD; ++it) {
            const int row = (it * GP_THREADS + tid) / (BN / 4), grow = m0 + row;
            float4 v = tile4(row, c * 16);
            const bool live = grow < M && gcol < N;
            if (EPI == 1 && !live) continue;
            v.x += old[it].x; v.y += old[it].y; v.z += old[it].z; v.w += old[it].w;
            if (live) *reinterpret_cast<float4*>(reinterpret_cast<float*>(Cv) + (size_t)grow * N + gcol) = v;
            if constexpr (EPI == 8) norm_out_row(v, gamma, live, grow, gcol, M, N, no);
        }
        return;
    }
    __syncthreads();
    if constexpr (EPI == 4) {
        // act = bf16(silu(g) * u) from the bf16-rounded g and u (the arithmetic of swiglu_rows_kernel / g2_swiglu_epilogue)
        constexpr int CH = BN / 16;                          // chunks of 8 act columns in a row
#pragma unroll
        for (int it = 0; it < (BM * CH + GP_THREADS - 1) / GP_THREADS; ++it) {
            const int item = it * GP_THREADS + tid, row = item / CH, c = item % CH;
            if (BM * CH % GP_THREADS != 0 && row >= BM) break;
            Vec<bf16> g, u;
            g.raw = *reinterpret_cast<const uint4*>(g2_smem + ct_off<ROWB>(row, c * 16));
            u.raw = *reinterpret_cast<const uint4*>(g2_smem + ct_off<ROWB>(row, BN + c * 16));
            float gf[8], uf[8];
            g.to_float(gf);
            u.to_float(uf);
#pragma unroll
            for (int e = 0; e < 8; ++e) gf[e] = gf[e] / (1.0f + __expf(-gf[e])) * uf[e];
            g.from_float(gf);
            const int grow = m0 + row, gcol = tn * (BN / 2) + c * 8;
            if (grow < M && gcol < N) g.store(reinterpret_cast<bf16*>(Cv) + (size_t)grow * N + gcol);
        }
    } else if constexpr (EPI == 3) {
        // the arithmetic of qknorm_rope_kvwrite_kernel on the bf16-rounded row, so the result is bit-identical to GEMM (bf16 store) + that kernel
        const int c = tid & 15;
        hr.finish(c, tn, m0 + hrow, 32, M, hd, reinterpret_cast<bf16*>(Cv), N, [&](int i, float (&x)[8]) {
            const int row = i * 32 + hrow;
            Vec<bf16> raw;
            raw.raw = *reinterpret_cast<const uint4*>(g2_smem + ct_off<ROWB>(row, c * 16));
            raw.to_float(x);
        });
    } else if constexpr (EPI == 2) {
        float* C = reinterpret_cast<float*>(Cv) + (size_t)blockIdx.y * M * N;
#pragma unroll
        for (int it = 0; it < BM * (BN / 4) / GP_THREADS; ++it) {
            const int item = it * GP_THREADS + tid, row = item / (BN / 4), c = item % (BN / 4);
            const float4 v = tile4(row, c * 16);
            const int grow = m0 + row, gcol = n0 + c * 4;
            if (grow < M && gcol < N) *reinterpret_cast<float4*>(C + (size_t)grow * N + gcol) = v;
        }
    } else if constexpr (EPI == 9) {
        constexpr int LN = BN / 4;                           // lanes that hold a row
#pragma unroll
        for (int it = 0; it < BM * LN / GP_THREADS; ++it) {
            const int item = it * GP_THREADS + tid, row = item / LN, c = item % LN;
            const float4 v = tile4(row, c * 16);
            const int grow = m0 + row, gcol = n0 + c * 4;
            const bool live = grow < M && gcol < N;
            if (live) *reinterpret_cast<float4*>(reinterpret_cast<float*>(Cv) + (size_t)grow * N + gcol) = v;
            float best = -INFINITY;                          // the lowest column of the largest value; NaN is never the best
            int at = 0x7FFFFFFF;
            if (live) {
                if (v.x > best) { best = v.x; at = gcol; }
                if (v.y > best) { best = v.y; at = gcol + 1; }
                if (v.z > best) { best = v.z; at = gcol + 2; }
                if (v.w > best) { best = v.w; at = gcol + 3; }
            }
#pragma unroll
            for (int off = LN / 2; off >= 1; off >>= 1) {
                const float ov = __shfl_xor(best, off, 64);
                const int oi = __shfl_xor(at, off, 64);
                if (ov > best || (ov == best && oi < at)) { best = ov; at = oi; }
            }
            if (c == 0 && grow < M) {
                bo.val[(size_t)grow * ntn + tn] = best;
                bo.idx[(size_t)grow * ntn + tn] = at;
            }
        }
    } else {
        // 8 columns per lane: two float4 -> 16 bytes of bf16
#pragma unroll
        for (int it = 0; it < BM * (BN / 8) / GP_THREADS; ++it) {
            const int item = it * GP_THREADS + tid, row = item / (BN / 8), c = item % (BN / 8);
            const float4 v0 = tile4(row, c * 32), v1 = tile4(row, c * 32 + 16);
            const int grow = m0 + row, gcol = n0 + c * 8;
            if (grow >= M || gcol >= N) continue;
            float f[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
            size_t orow = grow;
            if constexpr (EPI == 6) {
                orow = ga.order[grow];
                const float w = ga.wts[orow];
#pragma unroll
                for (int e = 0; e < 8; ++e) f[e] *= w;
            } else {
                if (bias) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) f[e] += to_f(bias[gcol + e]);
                }
                if constexpr (EPI == 5) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) f[e] = xielu<false>(f[e], xa.pos, xa.neg);
                }
                if constexpr (EPI == 7) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) f[e] = gelu_erf(f[e]);
                }
            }
            Vec<bf16> o;
            o.from_float(f);
            o.store(reinterpret_cast<bf16*>(Cv) + orow * N + gcol);
        }
    }
}
// The arguments up to `kps` arrive preloaded in SGPRs, 14 dwords (engine.hip, fused_gemv_kernel): what the first DMA waits for (the sign bit of kps: W is the packed copy), and
// the bias, which a plain product would otherwise ask for behind its loop: 129 rows, N = 4096, K = 1024 8.8 -> 8.7 us, with a bias, 300 rows, N = 3072 9.5 -> 9.4.
// (up to 128 x 128: two workgroups a CU, at most 80 KiB of LDS and 128 registers each - but for 128 x 64, whose ring of six takes 88 KiB; the larger ones have a CU to
// themselves)
template <int EPI, int WM, int WN>
__global__ __launch_bounds__(GP_THREADS, WM * WN <= 16 ? 4 : 2) void gemmp_bf16_kernel(const bf16* A, const bf16* W, void* Cv, const bf16* bias, int M, int N, int K, int ntm, int ntn, int kps,
                                                                       QkvHeadArgs hd, ActArgs xa, NormIn ni, NormOut no, BestOut bo) {
    gemmp_body<EPI, false, WM, WN>(A, W, bias, Cv, M, N, K, ntm, ntn, kps & INT_MAX, hd, (unsigned)kps >> 31, xa, GroupArgs{}, ni, no, bo);
}
template <int EPI>
__global__ __launch_bounds__(GP_THREADS, 4) void gemmp_grouped_kernel(const bf16* A, const bf16* W, bf16* C, int N, int K, int ntn, GroupArgs ga) {
    gemmp_body<EPI, true, 4, 4>(A, W, nullptr, C, 0, N, K, 0, ntn, K, QkvHeadArgs{}, 0, ActArgs{}, ga, NormIn{}, NormOut{}, BestOut{});
}

// ---- fp8 x fp8 with 128-wide block scales on the same structure --------------------------------------------
// K tile = 128 fp8 = one scale block: per tile the 256 row scales of A (fp32) and the two weight-block scales of
// the tile's 256 columns (bf16) are DMA'd into a small LDS array next to the operand tiles - every global load
// in the loop is an LDS-DMA, so no compiler-counted vmcnt ever drains the prefetch.  One v_mfma_f32_16x16x128_f8f6f4
// per 16x16 output tile and K tile, issued on a zero accumulator and folded in with the scale product.
__device__ __forceinline__ void g2_dma4(const void* src, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"(src), "s"(lds_addr) : "memory", "m0");
}
__device__ __forceinline__ void g2_dma2(const void* src, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_ushort %0, off" ::"v"(src), "s"(lds_addr) : "memory", "m0");
}

__device__ __forceinline__ void g2_dma4_so(const void* sbase, uint32_t voff, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(voff), "s"(sbase), "s"(lds_addr) : "memory", "m0");
}
__device__ __forceinline__ void g2_dma2_so(const void* sbase, uint32_t voff, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_ushort %0, %1" ::"v"(voff), "s"(sbase), "s"(lds_addr) : "memory", "m0");
}

constexpr int G2_SCALE_BYTES = 256 * 4 + 256;   // per buffer: 256 fp32 row scales | 64 lanes x 4 B of weight-scale slots (2 used)

template <int EPI>   // 0: bf16 C store; 1: fp32 C +=; 2: SwiGLU + e4m3 quantisation (W = fused gate / up rows, N = I; Cv = codes [M][I], Cs = scales [M][I/128]);
                     // 3: QKV heads (QkvHeadArgs; a tile holds two head slots)
__global__ __launch_bounds__(G2_THREADS) void gemm256_fp8_kernel(const uint8_t* A, const float* sa, const uint8_t* W, const bf16* sw,
                                                                  void* Cv, float* Cs, int M, int N, int K, int ntm, int ntn, QkvHeadArgs hd) {
    extern __shared__ __attribute__((aligned(16))) char g2_smem[];   // A[2] | W[2] | scales[2]
    const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);   // in an SGPR: it enters the DMAs' scalar bases
    const int wr = wid >> 2, wc = wid & 3, q = lane >> 4, l15 = lane & 15;
    int tm, tn;
    g2_tile_of(blockIdx.x, ntm * ntn, ntm, ntn, tm, tn);
    const int m0 = tm * G2_BM, n0 = tn * G2_BN;
    const int KB = K >> 7, NB = (N + 127) >> 7;

    // DMA sources as (uniform 64-bit base in SGPRs) + (per-lane 32-bit byte offset): 8 offset registers instead of 16
    // pointer registers in a kernel that lives at the 256-register line, and the per-K-tile advance is one scalar add.
    // Offsets are relative to the tile's first row (operand tiles span at most 255 rows x K <= 2^31 bytes).
    // LDS image: [256 rows][128 B], 16-byte chunk c of row r at position c ^ g2_sw8(r).  ds_read_b128 is served in the lane
    // groups {0-3, 12-15, 20-27}, {4-11, 16-19, 28-31} (+32) - not in runs of 16 lanes - and a fragment read has lanes (q =
    // lane >> 4, row lane & 15) fetch chunks 2 q / 2 q + 1: with the plain c ^ (r & 7) swizzle of the bf16 image, rows r and
    // r + 8 of such a group meet in the same banks (SQ_LDS_BANK_CONFLICT = 42 % of the LDS cycles of the first version);
    // XOR-ing 5 into the rows 8-15 of every 16 separates them for both reads (exhaustive check over the four lane groups).
    //
    // DMA sources: (wave-uniform 64-bit base in SGPRs) + (per-lane 32-bit byte offset).  Instruction i of a wave moves rows
    // 32 wid + 8 i + (lane >> 3); the row step 8 i K goes into the scalar base, so a lane needs TWO offsets for all eight
    // instructions of a stage (even / odd i differ in the swizzle only) - this kernel lives at the 256-register line, and
    // sixteen 64-bit source pointers (the first version) or eight offsets spill.  Whole tiles only: the caller sends shapes
    // with M % 256 or N % 256 != 0 to the 128-tile kernel (clamped row offsets are loop-invariant, so hipcc computes all
    // sixteen up front and spills them - and with them a few accumulators).
    // The per-lane offsets are RECOMPUTED from the lane id at every stage (a handful of vector instructions per tile): held
    // across the loop they are spilled at its fullest point, and every reload waits on the vector-memory counter.
    const uint8_t* a_tile = A + ((size_t)m0 + wid * 32) * K;
    // EPI 2: B-tile rows 0-127 = gate rows 128 tn .., rows 128-255 = up rows N + 128 tn .. (N = I): waves 0-3 stage gate rows, 4-7 up rows,
    // and the tile's two weight-scale blocks are block rows tn and I / 128 + tn
    const uint8_t* w_tile = W + (size_t)((EPI == 2) ? (wid < 4 ? tn * 128 + wid * 32 : N + tn * 128 + (wid - 4) * 32) : n0 + wid * 32) * K;
    const float* sa_tile = sa + ((size_t)m0 + (wid & 3) * 64) * KB;      // waves 0-3: 64 row scales each (one per lane)
    const bf16* sw_tile = sw + (size_t)((EPI == 2) ? tn : 2 * tn) * KB;  // wave 4: the tile's two weight-block scales (lanes 0 / 1)
    const uint32_t sw_step = (uint32_t)((EPI == 2) ? (N >> 7) : 1) * (uint32_t)(KB * 2);   // bytes between the two
    const uint32_t lds0 = g2_lds_addr(g2_smem);
    // operand tiles of K tile kt -> stage buf, as eight 1-KiB pieces (piece p: rows 8 (p >> 1) .. + 8 of this wave's 32, A for
    // even p, W for odd p).  Branch-free: the pieces are issued from the middle of the MFMA pipeline, one behind each MFMA of
    // a tile's last group - a DMA costs ~60 cycles of issue, which back to back (the first version) is ~500 cycles in which
    // neither wave of a SIMD issues an MFMA, and behind an MFMA mostly runs under it.
    auto stage_piece = [&](int kt, int buf, int p, uint32_t off_e, uint32_t off_o) {
        const int i = p >> 1;
        const uint32_t dst = __builtin_amdgcn_readfirstlane(lds0 + ((p & 1) ? 2 + buf : buf) * G2_TILE + wid * 4096 + i * 1024);
        const uint8_t* base = ((p & 1) ? w_tile : a_tile) + (size_t)kt * 128 + (size_t)8 * i * K;
        g2_dma16_so(base, (i & 1) ? off_o : off_e, dst);
    };
    auto stage_offsets = [&](uint32_t& off_e, uint32_t& off_o) {
        uint32_t ln = (uint32_t)lane;
        asm volatile("" : "+v"(ln));                                     // opaque: keeps the offsets out of the loop-invariant set
        const uint32_t r8 = ln >> 3, c8 = ln & 7;
        off_e = r8 * (uint32_t)K + ((c8 ^ r8) << 4);                     // rows 0-7 of 16: swizzle r & 7
        off_o = r8 * (uint32_t)K + ((c8 ^ r8 ^ 5u) << 4);                // rows 8-15: ^ 5 (g2_sw8)
    };
    auto stage = [&](int kt, int buf) {
        uint32_t off_e, off_o;
        stage_offsets(off_e, off_o);
#pragma unroll
        for (int p = 0; p < 8; ++p) stage_piece(kt, buf, p, off_e, off_o);
    };
    // scales of K tile kt -> scale stage buf (per-wave branches: issued at the top of a tile, outside the pipeline)
    auto stage_scales = [&](int kt, int buf) {
        const uint32_t s_dst = __builtin_amdgcn_readfirstlane(lds0 + 4 * G2_TILE + buf * G2_SCALE_BYTES + (wid < 4 ? wid * 256 : 1024));
        if (wid < 4) g2_dma4_so(sa_tile + kt, (uint32_t)lane * (uint32_t)(KB * 4), s_dst);
        else if (wid == 4) g2_dma2_so(sw_tile + kt, ((uint32_t)lane & 1u) * sw_step, s_dst);
    };

    f32x4_g acc[8][4];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_g{0.f, 0.f, 0.f, 0.f};

    // fragment reads: row = base + l15, the lane's 32 bytes are chunks 2q and 2q+1
    const int f_lo = l15 * 128 + (((2 * q) ^ g2_sw8(l15)) << 4);
    const int f_hi = l15 * 128 + (((2 * q + 1) ^ g2_sw8(l15)) << 4);
    const int a_base = wr * 128 * 128, w_base = wc * 64 * 128;

    // The MFMAs run as ONE software pipeline over the whole K loop, 32 per K tile (4 groups of 2 A row-tiles x 4 B column-tiles):
    // (1) the scale-and-add of product n is issued behind MFMA n + 2, every MFMA pinned by an empty volatile asm on its result:
    //     instruction selection otherwise sinks each product's FMAs directly under its own MFMA (s_nop 11 + two v_pk_fma per
    //     MFMA in the first version's ISA; sched_barrier only binds the later machine scheduler).  Scalar FMAs on purpose:
    //     beside MFMAs a v_pk_fma_f32 costs more issue time than the two v_fma_f32 it replaces;
    // (2) A fragments and row scales of group g + 1 are requested before group g's MFMAs;
    // (3) ONE barrier per K tile, at the start of its last group: by then every wave holds all fragments of tile kt in
    //     registers (stage kt & 1 is free) and its own share of tile kt + 1 - requested a whole tile earlier - has landed.
    //     Behind it the DMA of tile kt + 2 goes out, one piece behind each MFMA of the group, and the NEXT tile's first
    //     fragments are requested: group 0's A fragments at once, its row scales two steps later, each B fragment right
    //     after its last MFMA of this tile (the last group runs column-major for that).  No tile starts with an LDS round
    //     trip, a burst of DMA issue or a barrier.  Everything inside the pipeline is branch-free - one conditional DMA
    //     in it cut the basic block in two and made hipcc spill a hundred registers per tile - so the scales of tile
    //     kt + 1 (1 KiB under per-wave branches) are requested at the top of tile kt; their stage was last read in tile kt - 1.
    stage(0, 0);
    stage_scales(0, 0);
    stage(min(1, KB - 1), 1);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    i32x8_g fb[4], fa[2][2];
    f32x4_g t[3];
    f32x4_g sc[2][2];        // [slot][row-tile of the group]: raw row scales as they come from LDS, multiplied by the block scale in place
    float swv;
    uint32_t off_e = 0, off_o = 0;
    auto ldfrag = [&](const char* base) -> i32x8_g {
        const uint4 lo = *reinterpret_cast<const uint4*>(base + f_lo), hi = *reinterpret_cast<const uint4*>(base + f_hi);
        return i32x8_g{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
    };
    auto load_frags = [&](int buf, int g, int slot) {
        const char* As = g2_smem + buf * G2_TILE + a_base;
#pragma unroll
        for (int u = 0; u < 2; ++u) fa[slot][u] = ldfrag(As + (2 * g + u) * 2048);
    };
    // a group's row scales go into the slot the group BEFORE the previous one used: that one's last two scale-and-adds run
    // two steps into the next group, so the scales are requested at step 2 of a group, the fragments at step 0
    auto load_scales = [&](int buf, int g, int slot) {
        const char* Ss = g2_smem + 4 * G2_TILE + buf * G2_SCALE_BYTES;
#pragma unroll
        for (int u = 0; u < 2; ++u) sc[slot][u] = *reinterpret_cast<const f32x4_g*>(Ss + (wr * 128 + (2 * g + u) * 16 + q * 4) * 4);
    };
    // (a sub-dword LDS-DMA still strides the lanes by 4 bytes: lane l's 16 bits land at +4l, zero-extended)
    auto load_swv = [&](int buf) -> float { return to_f(*reinterpret_cast<const bf16*>(g2_smem + 4 * G2_TILE + buf * G2_SCALE_BYTES + 1024 + (wc >> 1) * 4)); };
#pragma unroll
    for (int j = 0; j < 4; ++j) fb[j] = ldfrag(g2_smem + 2 * G2_TILE + w_base + j * 2048);
    load_frags(0, 0, 0);
    load_scales(0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    // step n of a tile: group g = n / 8; groups 0-2 walk (row-tile u, column-tile j) row-major, group 3 column-major
#define G2F_U(N) (((N) < 24) ? (((N) >> 2) & 1) : ((N) & 1))
#define G2F_J(N) (((N) < 24) ? ((N) & 3) : (((N) & 7) >> 1))
#define G2F_FMA(NPREV)                                                                                              \
    {                                                                                                               \
        constexpr int g_ = (NPREV) >> 3, u_ = G2F_U(NPREV), j_ = G2F_J(NPREV), i_ = 2 * g_ + u_;                    \
        asm volatile("" : "+v"(t[(NPREV) % 3]));      /* ordered behind the MFMA issued just above (volatile asm statements keep their order) */ \
        _Pragma("unroll") for (int r = 0; r < 4; ++r) acc[i_][j_][r] = fmaf(t[(NPREV) % 3][r], sc[g_ & 1][u_][r], acc[i_][j_][r]); \
        __builtin_amdgcn_sched_barrier(0);                                                                          \
    }
#define G2F_STEP(N)                                                                                                 \
    {                                                                                                               \
        constexpr int g_ = (N) >> 3, u_ = G2F_U(N), j_ = G2F_J(N);                                                  \
        if constexpr ((N) == 24) {                                                                                  \
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");                                             \
            __builtin_amdgcn_s_barrier();                                                                           \
            stage_offsets(off_e, off_o);                                                                            \
            __builtin_amdgcn_sched_barrier(0);                                                                      \
        }                                                                                                           \
        if constexpr (((N) & 7) == 0) {                                                                             \
            if constexpr ((N) == 0) swv = load_swv(buf);                                                            \
            _Pragma("unroll") for (int u = 0; u < 2; ++u)                                                           \
                _Pragma("unroll") for (int r = 0; r < 4; ++r) sc[g_ & 1][u][r] *= swv;                              \
            __builtin_amdgcn_sched_barrier(0);                                                                      \
            if constexpr (g_ < 3) load_frags(buf, g_ + 1, (g_ + 1) & 1);                                            \
            else load_frags(buf ^ 1, 0, 0);                                                                         \
            __builtin_amdgcn_sched_barrier(0);                                                                      \
        }                                                                                                           \
        if constexpr (((N) & 7) == 2) {                                                                             \
            if constexpr (g_ < 3) load_scales(buf, g_ + 1, (g_ + 1) & 1);                                           \
            else load_scales(buf ^ 1, 0, 0);                                                                        \
            __builtin_amdgcn_sched_barrier(0);                                                                      \
        }                                                                                                           \
        t[(N) % 3] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fa[g_ & 1][u_], fb[j_], f32x4_g{0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0, 0, 0); \
        asm volatile("" : "+v"(t[(N) % 3]));          /* pins this MFMA here */                                     \
        __builtin_amdgcn_sched_barrier(0);                                                                          \
        if constexpr ((N) >= 24) {                    /* one DMA piece of tile kt + 2 behind each MFMA of the last group (past the end: re-reads the last tile into a stage nobody reads any more) */ \
            stage_piece(min(kt + 2, KB - 1), buf, (N) - 24, off_e, off_o);                                          \
            __builtin_amdgcn_sched_barrier(0);                                                                      \
        }                                                                                                           \
        if constexpr ((N) >= 24 && ((N) & 1) == 1) {  /* last use of column-tile j_ in this tile: fetch the next tile's */ \
            fb[j_] = ldfrag(g2_smem + (2 + (buf ^ 1)) * G2_TILE + w_base + j_ * 2048);                              \
            __builtin_amdgcn_sched_barrier(0);                                                                      \
        }                                                                                                           \
        if constexpr ((N) >= 2) G2F_FMA((N) - 2)                                                                    \
    }
    __builtin_amdgcn_s_setprio(1);
    for (int kt = 0; kt < KB; ++kt) {
        const int buf = kt & 1;
        stage_scales(min(kt + 1, KB - 1), buf ^ 1);
        G2F_STEP(0) G2F_STEP(1) G2F_STEP(2) G2F_STEP(3) G2F_STEP(4) G2F_STEP(5) G2F_STEP(6) G2F_STEP(7)
        G2F_STEP(8) G2F_STEP(9) G2F_STEP(10) G2F_STEP(11) G2F_STEP(12) G2F_STEP(13) G2F_STEP(14) G2F_STEP(15)
        G2F_STEP(16) G2F_STEP(17) G2F_STEP(18) G2F_STEP(19) G2F_STEP(20) G2F_STEP(21) G2F_STEP(22) G2F_STEP(23)
        G2F_STEP(24) G2F_STEP(25) G2F_STEP(26) G2F_STEP(27) G2F_STEP(28) G2F_STEP(29) G2F_STEP(30) G2F_STEP(31)
        G2F_FMA(30) G2F_FMA(31)
    }
    __builtin_amdgcn_s_setprio(0);
#undef G2F_STEP
#undef G2F_FMA
#undef G2F_U
#undef G2F_J
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");         // retire the phantom DMAs before the LDS is given back

    if constexpr (EPI == 2) {
        g2_swiglu_epilogue<true>(g2_smem, acc, tid, m0, tn, M, N, Cv, Cs);
        return;
    }
    if constexpr (EPI == 1) {     // N % 256 == 0 here
        g2_accum_epilogue(g2_smem, acc, tid, m0, n0, M, N, reinterpret_cast<float*>(Cv));
        return;
    }
    if constexpr (EPI == 3) {
        g2_qkv_heads_epilogue(g2_smem, acc, tid, m0, tn, M, N, reinterpret_cast<bf16*>(Cv), hd);
        return;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int col = n0 + wc * 64 + j * 16 + l15;
        if (col >= N) continue;
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = m0 + wr * 128 + i * 16 + q * 4 + r;
                if (row >= M) continue;
                if constexpr (EPI == 0) reinterpret_cast<bf16*>(Cv)[(size_t)row * N + col] = from_f<bf16>(acc[i][j][r]);
                else reinterpret_cast<float*>(Cv)[(size_t)row * N + col] += acc[i][j][r];
            }
    }
}

pgk_status gemm256_fp8_nt(const uint8_t* a, const float* sa, const uint8_t* w, const bf16* sw, void* c, bool accum_f32, int M, int N,
                          int K, hipStream_t st) {
    PGK_REQUIRE(K % 128 == 0 && K >= 128 && M % G2_BM == 0 && N % G2_BN == 0, "gemm256 fp8: M=%d N=%d must be multiples of 256 and K=%d of 128", M, N, K);
    constexpr size_t LDS = 4 * (size_t)G2_TILE + 2 * G2_SCALE_BYTES;
    static bool attr_done = false;
    if (!attr_done) {
        PGK_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm256_fp8_kernel<0>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS));
        PGK_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm256_fp8_kernel<1>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS));
        attr_done = true;
    }
    const int ntm = ceil_div(M, G2_BM), ntn = ceil_div(N, G2_BN);
    if (accum_f32) gemm256_fp8_kernel<1><<<ntm * ntn, G2_THREADS, LDS, st>>>(a, sa, w, sw, c, nullptr, M, N, K, ntm, ntn, QkvHeadArgs{});
    else gemm256_fp8_kernel<0><<<ntm * ntn, G2_THREADS, LDS, st>>>(a, sa, w, sw, c, nullptr, M, N, K, ntm, ntn, QkvHeadArgs{});
    PGK_CHECK_HIP(hipGetLastError());
    return PGK_OK;
}

// QKV projection finished per head in the epilogue (QkvHeadArgs): N = (Hq + 2 Hkv) x 128, two head slots per tile
pgk_status gemm256_fp8_qkv_heads_nt(const uint8_t* a, const float* sa, const uint8_t* w, const bf16* sw, bf16* qkv, int M, int N, int K,
                                    const QkvHeadArgs& hd, hipStream_t st) {
    PGK_REQUIRE(K % 128 == 0 && K >= 128 && M % G2_BM == 0 && N % G2_BN == 0 && N == (hd.hq + 2 * hd.hkv) * 128,
                "gemm256 fp8 qkv heads: M=%d, N=%d must be multiples of 256, K=%d of 128, N = (Hq + 2 Hkv) x 128", M, N, K);
    constexpr size_t LDS = 4 * (size_t)G2_TILE + 2 * G2_SCALE_BYTES;
    static bool attr_done = false;
    if (!attr_done) {
        PGK_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm256_fp8_kernel<3>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS));
        attr_done = true;
    }
    const int ntm = M / G2_BM, ntn = N / G2_BN;
    gemm256_fp8_kernel<3><<<ntm * ntn, G2_THREADS, LDS, st>>>(a, sa, w, sw, qkv, nullptr, M, N, K, ntm, ntn, hd);
    PGK_CHECK_HIP(hipGetLastError());
    return PGK_OK;
}

// act codes / scales = quantise(silu(a . Wg^T) * (a . Wu^T)), w = fused [2 I, K] gate / up codes with [2 I / 128][K / 128] block scales
pgk_status gemm256_fp8_swiglu_nt(const uint8_t* a, const float* sa, const uint8_t* w, const bf16* sw, uint8_t* q_out, float* s_out, int M,
                                 int I, int K, hipStream_t st) {
    PGK_REQUIRE(K % 128 == 0 && K >= 128 && M % G2_BM == 0 && I % 128 == 0, "gemm256 fp8 swiglu: M=%d must be a multiple of 256, I=%d and K=%d of 128", M, I, K);
    PGK_REQUIRE((const void*)a != (const void*)q_out, "gemm256 fp8 swiglu: output aliases the activation operand");
    constexpr size_t LDS = 4 * (size_t)G2_TILE + 2 * G2_SCALE_BYTES;
    static bool attr_done = false;
    if (!attr_done) {
        PGK_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm256_fp8_kernel<2>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS));
        attr_done = true;
    }
    const int ntm = M / G2_BM, ntn = I / 128;
    gemm256_fp8_kernel<2><<<ntm * ntn, G2_THREADS, LDS, st>>>(a, sa, w, sw, q_out, s_out, M, I, K, ntm, ntn, QkvHeadArgs{});
    PGK_CHECK_HIP(hipGetLastError());
    return PGK_OK;
}

// 192-column tiles when they fill the rounds of the chip better (cost = rounds x work per tile)
static bool gemm256_narrow(int M, int N) {
    const int ntm = ceil_div(M, G2_BM);
    return N % 192 == 0 && 0.75 * ceil_div(ntm * (N / 192), 256) < (double)ceil_div(ntm * ceil_div(N, G2_BN), 256) - 0.01;
}

// Of the kernels that finish SwiGLU or heads, the one whose lanes hold columns of a row (ct_off)
// where at most a tenth of the tiles' rows is padding, copies of the last row: they gain 0.3..1.8 % of a prompt there (ms, other way and this: Qwen3-0.6B, 3100 rows 6.03 / 5.91, 3500 6.49 / 6.38,
// 4096 7.27 / 7.20; Llama-3-8B shape, e4m3, 4096 49.9 / 49.7, bf16, 1500 and 2850 even), and lose where it is much: 300 rows, N = 28672, K = 4096, 90 us / 94.6.
static bool gemm256_rows(int M) { return 10LL * ((long long)ceil_div(M, G2_BM) * G2_BM - M) <= M; }
// Of the kernels that store from registers likewise, and only where a lane's four columns are one 8-byte store: stored one by one they are 16 rows to an instruction instead of 4.
// Us of pgk_gemm_nt, by columns / by rows: 4096 rows, N = K = 4096, C four bytes off a line 116 / 123, N = 4097 174 / 196, 3000 rows, N = 50257, K = 1024 395 / 484;
// whole and aligned, 4096 rows, N = 4100 173 / 167, 3000 rows, N = 50256, K = 1024 377 / 346, 512 rows, N = 32768, K = 1024 40.8 / 36.8; padding: 300 rows, N = 28672, K = 4096
// 90 / 99, 600 171 / 178, 257 rows, N = 32768, K = 1024 31.4 / 35, 1100 rows, N = 12288, K = 4096 even.
static bool gemm256_rows_store(int M, int N, const void* C) { return gemm256_rows(M) && N % 4 == 0 && ((uintptr_t)C & 7) == 0; }

// QKV projection finished head by head: where whole 256-column tiles are what gemm256_bf16_nt would take
bool gemm256_bf16_qkv_heads_ok(int M, int N, int K) { return K % 64 == 0 && K >= 64 && N % 256 == 0 && !gemm256_narrow(M, N); }
pgk_status gemm256_bf16_qkv_heads_nt(const bf16* A, const bf16* W, bf16* qkv, int M, int N, int K, const QkvHeadArgs& hd, hipStream_t st, bool packed, const NormIn& ni) {
    PGK_REQUIRE(gemm256_bf16_qkv_heads_ok(M, N, K) && N == (hd.hq + 2 * hd.hkv) * 128, "gemm256 heads: N=%d K=%d (%d + 2 x %d heads)", N, K, hd.hq, hd.hkv);
    static bool attr_done = false;
    if (!attr_done) {
        for (auto* kfn : {&gemm256s_bf16_kernel<5>, &gemm256s_bf16_kernel<5, 4, true>})
            PGK_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kfn), hipFuncAttributeMaxDynamicSharedMemorySize, (int)G2S_LDS));
        attr_done = true;
    }
    const int ntm = ceil_div(M, G2_BM), ntn = N / G2_BN;
    auto kfn = gemm256_rows(M) ? &gemm256s_bf16_kernel<5, 4, true> : &gemm256s_bf16_kernel<5>;
    kfn<<<ntm * ntn, G2_THREADS, G2S_LDS, st>>>(A, W, nullptr, qkv, M, N, K, ntm, ntn, packed ? 1 : 0, ActArgs{}, hd, ni);
    PGK_CHECK_HIP(hipGetLastError());
    return PGK_OK;
}

// bf16 NT on the 256^2 structure; caller guarantees K % 64 == 0 and 16-byte aligned rows
pgk_status gemm256_bf16_nt(const bf16* A, const bf16* W, const bf16* bias, void* C, bool accum_f32, int M, int N, int K,
                           hipStream_t st, bool packed, const ActArgs* act, const NormIn& ni) {
    PGK_REQUIRE(K % 64 == 0 && K >= 64, "gemm256: K=%d must be a multiple of 64", K);
    PGK_REQUIRE(!packed || N % 16 == 0, "gemm256: the fragment-major weight copy has whole 16-row tiles (N=%d)", N);
    constexpr size_t LDS = G2S_LDS;
    static bool attr_done = false;
    if (!attr_done) {
        PGK_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm256_bf16_kernel<0>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS));
        PGK_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm256_bf16_kernel<1>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS));
        attr_done = true;
    }
    const int ntm = ceil_div(M, G2_BM), ntn = ceil_div(N, G2_BN);
    const char* e = getenv("PGK_GEMM256S");          // 0: two full stages, waves in lockstep; default: staggered phases
    if (packed || act || ni.ss || !e || atoi(e) != 0) {
        static bool attr_s = false;
        if (!attr_s) {
            for (auto* kfn : {&gemm256s_bf16_kernel<0>, &gemm256s_bf16_kernel<0, 4, true>, &gemm256s_bf16_kernel<0, 3>, &gemm256s_bf16_kernel<0, 3, true>, &gemm256s_bf16_kernel<1>})
                PGK_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kfn), hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS));
            attr_s = true;
        }
        const bool narrow = !accum_f32 && gemm256_narrow(M, N), rows = gemm256_rows_store(M, N, C);
        const int nt = narrow ? N / 192 : ntn;
        if (act) {
            auto pick = [&](auto epi) {
                constexpr int E = decltype(epi)::value;
                if (narrow) return rows ? &gemm256s_bf16_kernel<E, 3, true> : &gemm256s_bf16_kernel<E, 3>;
                return rows ? &gemm256s_bf16_kernel<E, 4, true> : &gemm256s_bf16_kernel<E>;
            };
            auto kfn = act->gelu ? pick(std::integral_constant<int, 4>{}) : pick(std::integral_constant<int, 3>{});
            static bool attr_x[2][2][2] = {};
            bool& done = attr_x[act->gelu][narrow][rows];
            if (!done) PGK_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kfn), hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS));
            done = true;
            kfn<<<ntm * nt, G2_THREADS, LDS, st>>>(A, W, nullptr, C, M, N, K, ntm, nt, packed ? 1 : 0, *act, QkvHeadArgs{}, NormIn{});
        } else if (accum_f32) gemm256s_bf16_kernel<1><<<ntm * ntn, G2_THREADS, LDS, st>>>(A, W, nullptr, C, M, N, K, ntm, ntn, packed ? 1 : 0, ActArgs{}, QkvHeadArgs{}, NormIn{});
        else {
            auto kfn = narrow ? (rows ? &gemm256s_bf16_kernel<0, 3, true> : &gemm256s_bf16_kernel<0, 3>) : rows ? &gemm256s_bf16_kernel<0, 4, true> : &gemm256s_bf16_kernel<0>;
            kfn<<<ntm * nt, G2_THREADS, LDS, st>>>(A, W, bias, C, M, N, K, ntm, nt, packed ? 1 : 0, ActArgs{}, QkvHeadArgs{}, ni);
        }
        PGK_CHECK_HIP(hipGetLastError());
        return PGK_OK;
    }
    if (accum_f32) gemm256_bf16_kernel<1><<<ntm * ntn, G2_THREADS, LDS, st>>>(A, W, nullptr, C, M, N, K, ntm, ntn);
    else gemm256_bf16_kernel<0><<<ntm * ntn, G2_THREADS, LDS, st>>>(A, W, bias, C, M, N, K, ntm, ntn);
    PGK_CHECK_HIP(hipGetLastError());
    return PGK_OK;
}

// act[M][I] = bf16(silu(A . Wg^T) * (A . Wu^T)), W = fused [2 I, K] gate / up weight (staggered kernel, SwiGLU epilogue)
pgk_status gemm256_bf16_swiglu_nt(const bf16* A, const bf16* W, bf16* act, int M, int I, int K, hipStream_t st, bool packed, const NormIn& ni) {
    PGK_REQUIRE(K % 64 == 0 && K >= 64 && I % 128 == 0, "gemm256 swiglu: K=%d must be a multiple of 64 and I=%d of 128", K, I);
    constexpr size_t LDS = G2S_LDS;
    static bool attr_done = false;
    if (!attr_done) {
        for (auto* kfn : {&gemm256s_bf16_kernel<2>, &gemm256s_bf16_kernel<2, 3>, &gemm256s_bf16_kernel<2, 4, true>, &gemm256s_bf16_kernel<2, 3, true>})
            PGK_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kfn), hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS));
        attr_done = true;
    }
    const bool rows = gemm256_rows(M);
    const int ntm = ceil_div(M, G2_BM), ntn = I / 128;
    // 96 act columns per tile (192-column B tiles) when that fills the rounds of the chip better: Qwen3-0.6B at S = 2048 is
    // 8 x 24 = 192 tiles of 128 (three quarters of the CUs, one round) or 8 x 32 = 256 tiles of 96 (all of them)
    if (I % 96 == 0 && 0.75 * ceil_div(ntm * (I / 96), 256) < (double)ceil_div(ntm * ntn, 256) - 0.01) {
        auto kfn = rows ? &gemm256s_bf16_kernel<2, 3, true> : &gemm256s_bf16_kernel<2, 3>;
        kfn<<<ntm * (I / 96), G2_THREADS, LDS, st>>>(A, W, nullptr, act, M, I, K, ntm, I / 96, packed ? 1 : 0, ActArgs{}, QkvHeadArgs{}, ni);
    } else {
        auto kfn = rows ? &gemm256s_bf16_kernel<2, 4, true> : &gemm256s_bf16_kernel<2>;
        kfn<<<ntm * ntn, G2_THREADS, LDS, st>>>(A, W, nullptr, act, M, I, K, ntm, ntn, packed ? 1 : 0, ActArgs{}, QkvHeadArgs{}, ni);
    }
    PGK_CHECK_HIP(hipGetLastError());
    return PGK_OK;
}

template <int EPI, int WM, int WN>
static pgk_status gemmp_launch(const bf16* A, const bf16* W, const bf16* bias, void* C, int M, int N, int K, int kps, const QkvHeadArgs& hd, int packed, const ActArgs& xa,
                               const NormIn& ni, const NormOut& no, hipStream_t st, const BestOut& bo = BestOut{}) {
    constexpr size_t LDS = gemmp_lds<EPI, WM, WN>();
    static bool attr_done = false;
    if (!attr_done) {
        PGK_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&gemmp_bf16_kernel<EPI, WM, WN>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS));
        attr_done = true;
    }
    const int ntm = ceil_div(M, 32 * WM), ntn = EPI == 4 ? ceil_div(N, 16 * WN) : ceil_div(N, 32 * WN);      // SwiGLU: N = I act columns, half a tile's
    gemmp_bf16_kernel<EPI, WM, WN><<<dim3(ntm * ntn, ceil_div(K, kps)), GP_THREADS, LDS, st>>>(A, W, C, bias, M, N, K, ntm, ntn, packed ? kps | INT_MIN : kps, hd, xa, ni, no, bo);
    PGK_CHECK_HIP(hipGetLastError());
    return PGK_OK;
}

// Tile of a product of `cols` weight rows in `splits` runs of K: the cheapest by rounds of workgroups x (time of a stage x stages + start and epilogue), in 0.01 us for
// one and, where the LDS lets it, for two workgroups on a CU.  The prices rank the tiles and are not a launch's time, which is 1.2 to 1.4 times as
// long.  `most`: how far down the list the product's epilogue goes (QKV heads are 128 columns, split products leave most
// of a round idle anyway).  Us a launch, K = 1024, measured (priced): 384 rows, N = 4096 10.1 (8.4) on 128 x 128, 8.4 (6.2) on 64 x 128; 93 rows, N = 6144 9.8 (8.4),
// 7.5 (6.2), 6.3 (5.0) on 64 x 64; 1531 rows, N = 4096 18.7 (13.5) on 128 x 128, 16.6 (12.1) on 192 x 128, N = 6144 27.8 (21.8) on 128 x 128, 23.0 (17.4) on 192 x 192.
enum { GP_128, GP_64_128, GP_192_128, GP_192, GP_64 };
static int gemmp_tile(int M, int cols, int K, int splits, int most) {
    constexpr struct { int bm, bn, one, one_fixed, two, two_fixed; } t[] = {{128, 128, 18, 260, 29, 420}, {64, 128, 13, 200, 20, 330}, {192, 128, 27, 350, 0, 0}, {192, 192, 40, 460, 0, 0}, {64, 64, 11, 150, 16, 260}};
    int best = 0;
    long long least = 0;
    for (int i = 0; i <= most; ++i) {
        const long long n = (long long)ceil_div(M, t[i].bm) * ceil_div(cols, t[i].bn) * splits, stages = K / splits / 32;
        const long long one = stages * t[i].one + t[i].one_fixed, two = stages * t[i].two + t[i].two_fixed;
        const long long cost = t[i].two ? n / 512 * two + (n % 512 > 256 ? two : n % 512 > 0 ? one : 0) : ceil_div(n, 256LL) * one;
        if (i == 0 || cost < least) { best = i; least = cost; }
    }
    return best;
}

// The same for a product that ends in the residual epilogue with a norm (nothing of it splits along K, so few rows ask for small tiles).
// 0: 128 x 128, 1: 128 x 64, 2: 64 x 64, 3: 96 x 64, 4: 32 x 64; two workgroups on a CU for 0, 2 and 4.
// Ms a prompt of Qwen3-0.6B with 1, 2, 3, 4: 450 rows 1.95 / 1.73 / 1.93 / 1.66, 600 2.20 / 1.98 / 2.07 / 2.08, 800 2.39 / 2.25 / 2.32 / 2.37, 1100 2.80 / 2.84 / 2.77 / 2.91,
// 1531 3.14 / 3.20 / 3.06 / 3.41, 1800 3.55 / 3.75 / 3.81 / 4.08.
// The prices of 64 x 64 and 96 x 64 are from before K was split over their waves, and 96 x 64 is priced for one workgroup a CU though two fit.  What they choose is within 0.4 % of the best tile at 14 lengths
// from 140 to 2600 rows of Qwen3-0.6B and at 8 of widths 1536 to 3072, but for 2100 rows (96 x 64 would take 4.34 ms, 128 x 128 takes 4.39) and width 3072 at 300 and 700 rows (1.28 / 1.29, 1.96 / 2.07).
static int gemmp_resid_tile(int M, int N, int K, int* cost) {
    constexpr struct { int bm, bn, one, one_fixed, two, two_fixed; } t[] = {{128, 128, 18, 450, 29, 640}, {128, 64, 14, 400, 0, 0}, {64, 64, 11, 300, 16, 400}, {96, 64, 13, 350, 0, 0}, {32, 64, 8, 250, 13, 350}};
    int best = 0;
    for (int i = 0; i < 5; ++i) {
        const long long n = (long long)ceil_div(M, t[i].bm) * ceil_div(N, t[i].bn), stages = K / 32;
        const long long one = stages * t[i].one + t[i].one_fixed, two = stages * t[i].two + t[i].two_fixed;
        const long long c = t[i].two ? n / 512 * two + (n % 512 > 256 ? two : n % 512 > 0 ? one : 0) : ceil_div(n, 256LL) * one;
        if (i == 0 || c < *cost) { best = i; *cost = (int)(c < INT_MAX ? c : INT_MAX); }
    }
    return best;
}
// Whether that epilogue pays against a product in `splits` slabs (or `splits` = 1, fp32 +=) and the norm's pass, which takes 6 us and a launch, less what
// the scaled rows cost the next product.  Qwen3-0.6B, us with the norm, before the small tiles split K: 1531 rows o 20.7 / 14.5, down 25 / 20; 384 rows 15 / 11, 17.5 / 14.5.
bool gemm128s_resid_pays(int M, int N, int K, int splits) {
    if (N % 64 != 0) return false;
    if (splits == 1) return true;
    int cost;
    gemmp_resid_tile(M, N, K, &cost);
    return cost <= K / splits / 32 * 18 + 260 + 720;
}

// mode 0: bf16 C (+bias, or with `act` its activation), 1: fp32 C +=, 2: fp32 slabs [splits][M][N] (K split into `splits` runs of whole 64-k steps),
// 3: QKV heads, 4: SwiGLU, 5: 1 with what the next RMSNorm leaves to do (NormOut); 0, 3, 4: rows scaled by NormIn where given
bool gemm128s_shape_ok(int N, int K) { return K % 64 == 0 && K >= 64 && N % 8 == 0 && N >= 8; }
bool gemm128s_ok(int M, int N, int K) { return M > 128 && gemm128s_shape_ok(N, K); }
pgk_status gemm128s_bf16_nt(const bf16* A, const bf16* W, const bf16* bias, void* C, int mode, int splits, int M, int N, int K, hipStream_t st,
                            const QkvHeadArgs* heads, bool packed, const ActArgs* act, const NormIn& ni, const NormOut& no) {
    PGK_REQUIRE(!packed || N % 16 == 0, "gemm128s: the fragment-major weight copy has whole 16-row tiles (N=%d)", N);
    const int pk = packed ? 1 : 0;
    PGK_REQUIRE(M >= 1 && gemm128s_shape_ok(N, K) && mode >= 0 && mode <= 5 && splits >= 1 && (splits == 1 || mode == 2), "gemm128s: M=%d N=%d K=%d mode=%d splits=%d", M, N, K, mode, splits);
    PGK_REQUIRE(mode != 4 || N % 64 == 0, "gemm128s: the SwiGLU epilogue needs I=%d to be a multiple of 64", N);
    PGK_REQUIRE(mode != 3 || (heads && N == (heads->hq + 2 * heads->hkv) * 128), "gemm128s: the QKV-heads epilogue needs N=%d = (Hq + 2 Hkv) x 128", N);
    PGK_REQUIRE(mode != 5 || (N % 64 == 0 && no.gamma && no.x && no.ss), "gemm128s: the residual epilogue with a norm needs N=%d to be a multiple of 64", N);
    PGK_REQUIRE(!ni.ss || (!ni.ld && (mode == 0 || mode == 3 || mode == 4)), "gemm128s: mode %d does not scale its rows", mode);
    const QkvHeadArgs hd = heads ? *heads : QkvHeadArgs{};
    const int kps = ceil_div(ceil_div(K, splits), 64) * 64;
    PGK_REQUIRE(ceil_div(K, kps) == splits, "gemm128s: K=%d does not split into %d runs of whole 64-k steps", K, splits);
    const ActArgs none{};
    if (mode == 0 && act && act->gelu) return gemmp_launch<7, 4, 4>(A, W, nullptr, C, M, N, K, kps, hd, pk, *act, ni, no, st);
    if (mode == 0 && act) return gemmp_launch<5, 4, 4>(A, W, nullptr, C, M, N, K, kps, hd, pk, *act, ni, no, st);
    if (mode == 0) return gemmp_launch<0, 4, 4>(A, W, bias, C, M, N, K, kps, hd, pk, none, ni, no, st);
    if (mode == 1) return gemmp_launch<1, 4, 4>(A, W, nullptr, C, M, N, K, kps, hd, pk, none, ni, no, st);
    if (mode == 2) {
        if (gemmp_tile(M, N, K, splits, GP_64_128) == GP_64_128) return gemmp_launch<2, 2, 4>(A, W, nullptr, C, M, N, K, kps, hd, pk, none, ni, no, st);
        return gemmp_launch<2, 4, 4>(A, W, nullptr, C, M, N, K, kps, hd, pk, none, ni, no, st);
    }
    if (mode == 5) {
        int cost;
        const int t = gemmp_resid_tile(M, N, K, &cost);
        if (t == 1) return gemmp_launch<8, 4, 2>(A, W, nullptr, C, M, N, K, kps, hd, pk, none, ni, no, st);
        if (t == 2) return gemmp_launch<8, 2, 2>(A, W, nullptr, C, M, N, K, kps, hd, pk, none, ni, no, st);
        if (t == 3) return gemmp_launch<8, 3, 2>(A, W, nullptr, C, M, N, K, kps, hd, pk, none, ni, no, st);
        if (t == 4) return gemmp_launch<8, 1, 2>(A, W, nullptr, C, M, N, K, kps, hd, pk, none, ni, no, st);
        return gemmp_launch<8, 4, 4>(A, W, nullptr, C, M, N, K, kps, hd, pk, none, ni, no, st);
    }
    if (mode == 3) {
        const int t = gemmp_tile(M, N, K, 1, GP_192_128);
        if (t == GP_64_128) return gemmp_launch<3, 2, 4>(A, W, nullptr, C, M, N, K, kps, hd, pk, none, ni, no, st);
        if (t == GP_192_128) return gemmp_launch<3, 6, 4>(A, W, nullptr, C, M, N, K, kps, hd, pk, none, ni, no, st);
        return gemmp_launch<3, 4, 4>(A, W, nullptr, C, M, N, K, kps, hd, pk, none, ni, no, st);
    }
    const int t = gemmp_tile(M, 2 * N, K, 1, GP_64);
    if (t == GP_64_128) return gemmp_launch<4, 2, 4>(A, W, nullptr, C, M, N, K, kps, hd, pk, none, ni, no, st);
    if (t == GP_192_128) return gemmp_launch<4, 6, 4>(A, W, nullptr, C, M, N, K, kps, hd, pk, none, ni, no, st);
    if (t == GP_192) return gemmp_launch<4, 6, 6>(A, W, nullptr, C, M, N, K, kps, hd, pk, none, ni, no, st);
    if (t == GP_64) return gemmp_launch<4, 2, 2>(A, W, nullptr, C, M, N, K, kps, hd, pk, none, ni, no, st);
    return gemmp_launch<4, 4, 4>(A, W, nullptr, C, M, N, K, kps, hd, pk, none, ni, no, st);
}

// act[M][I] = SwiGLU of few rows (a prompt of up to 128, the step of a batch) against the fragment-major gate / up copy: 64 x 64 tiles, 32 act columns each.  The
// packed kernel gives a wave the weights in registers and a workgroup 32 rows: us a launch there / here, K = 1024, I = 3072: 93 rows 10.9 / 7.8, 64 rows 8.5 / 7.3,
// 37 rows 8.1 / 7.2; ms, 4 steps of 24 sequences 4.07 / 3.97, a prompt of 9 1.083 / 1.051.  Smaller weights stay there, where more workgroups start earlier: us a layer there / here, K = 512,
// I = 1024 1 row 28.3 / 29.2, 96 rows 32.4 / 32.7; K = 1024, I = 2048 9 rows 32.9 / 33.4, 96 rows 38.4 / 38.6; but I = 3072 9 rows 35.0 / 34.3, 96 rows 41.1 / 39.5, and K = 1536, I = 1024
// 9 rows 46.9 / 45.8, 96 rows 50.1 / 49.5.
bool gemm_few_swiglu_ok(int I, int K) { return K % 64 == 0 && I % 32 == 0 && (K >= 1536 || (K >= 1024 && I >= 3072)); }
pgk_status gemm_few_swiglu_nt(const bf16* A, const bf16* wp, bf16* act, int M, int I, int K, const NormIn& ni, hipStream_t st) {
    PGK_REQUIRE(M >= 1 && gemm_few_swiglu_ok(I, K) && (!ni.ss || (ni.ld == 64 && ni.n <= 64)), "gemm_few_swiglu: M=%d I=%d K=%d", M, I, K);
    return gemmp_launch<4, 2, 2>(A, wp, nullptr, act, M, I, K, K, QkvHeadArgs{}, 1, ActArgs{}, ni, NormOut{}, st);
}

// Logits of a batch's step against the fragment-major lm_head: 64 x 128 tiles, bound by the stream of the weights and the fp32 rows (5.6 TB/s at 64 rows).  The kernel of
// 16 columns a workgroup stores 64 bytes of a row at a time; here 512.  K = 1024, 151936 columns, us a launch there / here: 64 rows 82 / 62; us a step
// of Qwen3-0.6B: 64 sequences 1172 / 1154, 48 1118 / 1104, 33 1093 / 1084, 24 1030 / 1029, 17 1011 / 1013: from 33 on.  From 64 tiles of columns on: 33 and 64 sequences, 4096 columns
// 136.0 / 137.3 and 140.3 / 140.4, 8192 139.5 / 137.3 and 145.2 / 140.5.
constexpr int GP_LOGITS_COLS = 128;
bool gemm_few_logits_ok(int M, int V, int K) { return M > 32 && V >= 64 * GP_LOGITS_COLS && K % 64 == 0 && K >= 64 && V % 16 == 0; }
int gemm_few_logits_blocks(int V) { return ceil_div(V, GP_LOGITS_COLS); }     // parts per row of best_val and best_idx
pgk_status gemm_few_logits_nt(const bf16* A, const bf16* wp, float* logits, float* best_val, int* best_idx, int M, int V, int K, hipStream_t st) {
    PGK_REQUIRE(gemm_few_logits_ok(M, V, K) && best_val && best_idx, "gemm_few_logits: M=%d V=%d K=%d", M, V, K);
    return gemmp_launch<9, 2, GP_LOGITS_COLS / 32>(A, wp, nullptr, logits, M, V, K, K, QkvHeadArgs{}, 1, ActArgs{}, NormIn{}, NormOut{}, st, BestOut{best_val, best_idx});
}

template <int EPI>
static pgk_status gemmp_grouped_launch(const bf16* A, const bf16* W, bf16* C, const GroupArgs& g, int max_tiles, int ntn, int N, int K, hipStream_t st) {
    constexpr size_t LDS = gemmp_lds<EPI, 4, 4>();
    static bool attr_done = false;
    if (!attr_done) {
        PGK_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&gemmp_grouped_kernel<EPI>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS));
        attr_done = true;
    }
    gemmp_grouped_kernel<EPI><<<max_tiles * ntn, GP_THREADS, LDS, st>>>(A, W, C, N, K, ntn, g);
    PGK_CHECK_HIP(hipGetLastError());
    return PGK_OK;
}
pgk_status gemm128s_grouped(const bf16* A, const bf16* W, bf16* C, MoeProduct what, const GroupArgs& g, int max_tiles, int rows, int N, int K, hipStream_t st) {
    PGK_REQUIRE(K % 64 == 0 && N % 64 == 0 && max_tiles >= 1 && g.tiles && g.n_tiles && g.order && g.wts, "gemm128s_grouped: N=%d K=%d", N, K);
    const int ntn = what == MOE_SWIGLU ? N / 64 : ceil_div(N, 128);
    if (what == MOE_GELU) return gemmp_grouped_launch<7>(A, W, C, g, max_tiles, ntn, N, K, st);
    if (what == MOE_DOWN) return gemmp_grouped_launch<6>(A, W, C, g, max_tiles, ntn, N, K, st);
    return gemmp_grouped_launch<4>(A, W, C, g, max_tiles, ntn, N, K, st);
}

}  // namespace pgk
