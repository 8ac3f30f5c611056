// Decode attention of a batch, streamed through the matrix pipe; included by engine.hip behind AttnArgs.
//
// attn_decode_kernel scores with dot2 instructions and reduces across 16 lanes per position: with two query heads per key head it issues 30-40
// vector instructions for every KiB of cache, and one slice per sequence left a batch of mixed contexts waiting for its longest (37 sequences of
// 200..3900 positions, 311 MB of cache per layer: 91 us; now 60, 5.2 TB/s).  Here a workgroup is one slice of one (sequence, key head) and each of its 4 waves
// streams groups of 32 positions on its own:
//   * a lane keeps the next group in registers (16 loads of 1 KiB contiguous per wave: 64 KiB in flight per workgroup, three of them per CU)
//     while the wave turns the present one into operands through 8 KiB of its own LDS, no barrier in the loop;
//   * S^T = K Q^T, the query heads of the key head as columns (any group of up to 16: one launch where groups other than 1, 2, 4 took several);
//     softmax lane-local; O^T += V^T P^T with V read through the transposing LDS read (the scheme of attn_oproj_mfma_kernel);
//   * the position is known before the first row is requested: slices beyond a sequence's context cost nothing, and no byte is read in vain
//     (requesting the first rows before it, as attn_decode_kernel does, was 2 % slower per step for 40 sequences of 60 positions).
// q is rounded to bf16 scaled, the probabilities to bf16, everything else is fp32: as the kernels it replaces.
#pragma once

// (row, 16-byte chunk) -> byte offset of a group's image; D = 64 packs two rows per 256 bytes
template <int D> __device__ __forceinline__ int as_koff(int row, int ch) { return row * (2 * D) + ((ch ^ (D == 128 ? row & 15 : (row >> 1) & 7)) << 4); }
template <int D> __device__ __forceinline__ int as_voff(int row, int ch) {
    const int x = D == 128 ? ((row & 3) << 2) | ((row >> 2) & 3) : (((row >> 1) & 1) << 2) | ((row >> 2) & 3);
    return row * (2 * D) + ((ch ^ x) << 4);
}

constexpr int AS_WAVES = 4, AS_GROUP = 32, AS_HEADS = 16;
template <int D> constexpr int as_image() { return AS_GROUP * 2 * D; }
template <int D> inline size_t as_lds(int G) {
    const size_t states = (size_t)AS_WAVES * G * (D + 4) * 4, images = (size_t)AS_WAVES * as_image<D>();
    return states > images ? states : images;
}

// grid (Hkv, slices, batch), the key head fastest: workgroups are dealt to the XCDs in turn, and with eight slices fastest the first slices, which
// every sequence has, all went to one XCD.  Slice s holds cache rows [s * chunk, (s + 1) * chunk), the last one to the end of the context.  DIRECT: one slice,
// normalised output; otherwise records (m, l, o) for attn_merge_kernel.
template <int D, bool DIRECT>
__global__ __launch_bounds__(256, 3) void attn_stream_kernel(unsigned long long* tl, AttnArgs a, int chunk) {
    const TLStamp tls(tl);
    typedef __bf16 bf16x8_s __attribute__((ext_vector_type(8)));
    typedef float f32x4_s __attribute__((ext_vector_type(4)));
    typedef short v4s_s __attribute__((ext_vector_type(4)));
    constexpr int LPR = D / 8, KS = D / 32, DT = D / 16, RS = D + 4, RPI = 64 / LPR, NI = AS_GROUP / RPI;   // lanes per row, k-steps, dim tiles, rows and loads
    extern __shared__ __attribute__((aligned(16))) char as_smem[];
    __shared__ __attribute__((aligned(16))) uint4 q_sh[AS_HEADS][LPR], kv_sh[2][LPR];
    __shared__ float s_new[AS_HEADS];
    const int G = a.g_total;
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l15 = lane & 15, q4 = lane >> 4;
    const int kvh = blockIdx.x, b = blockIdx.z, nsl = gridDim.y, slice = (int)((blockIdx.y + b) % (unsigned)nsl);
    const size_t head_off = ((size_t)b * a.hkv + kvh) * a.max_seq * D;
    const bf16* kc = a.kcache + head_off;
    const bf16* vc = a.vcache + head_off;
    uint4 kr[NI], vr[NI];
    auto at = [&](const bf16* base, int g0, int i, int ln, int end) {
        const uint32_t off = (uint32_t)min(g0 + i * RPI + ln / LPR, end) * (2 * D) + (ln % LPR) * 16;
        return *reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(base) + off);
    };
    const int pos = load_uniform_i32(a.positions + b);
    const int ctx = min(pos + 1, a.max_seq);
    const int c0 = DIRECT ? 0 : slice * chunk;
    const bool last = DIRECT || slice == nsl - 1;
    float* rec = DIRECT ? nullptr : a.part + (((size_t)b * a.hq + (size_t)kvh * G) * a.nsplit + slice) * (D + 2);
    if (!DIRECT && c0 >= ctx) {                                  // workgroup-uniform
        for (int e = threadIdx.x; e < G * (D + 2); e += 256) rec[(size_t)(e / (D + 2)) * a.nsplit * (D + 2) + e % (D + 2)] = e % (D + 2) ? 0.f : -INFINITY;
        tls.end();
        return;
    }
    const bool owns_new = pos < a.max_seq && pos >= c0 && (last || pos < c0 + chunk);
    const int c1 = min(last ? ctx : min(c0 + chunk, ctx), min(pos, a.max_seq));   // cached rows of the slice end here; the new token's comes from registers

    // ---- the new token: vector `item` (query heads, key, value) of 16 per pass to LPR lanes ----
    constexpr int IPW = 64 / LPR;                                // items per wave and pass
    const int sub = lane % LPR, ig = wid * IPW + lane / LPR;
    const float* row = a.qkv + (size_t)b * a.qkv_ld;
    auto item_off = [&](int it) { return it < G ? (kvh * G + it) * D : (it == G ? a.hq + kvh : a.hq + a.hkv + kvh) * D; };
    const int it0 = min(ig, G + 1);
    const float4 x0 = *reinterpret_cast<const float4*>(row + item_off(it0) + sub * 8), x1 = *reinterpret_cast<const float4*>(row + item_off(it0) + sub * 8 + 4);
    const int dd = (sub * 8) % (D / 2);
    const float* cp = a.rope_cos + (size_t)b * (D / 2) + dd;
    const float* sp = a.rope_sin + (size_t)b * (D / 2) + dd;
    const float4 cs0 = *reinterpret_cast<const float4*>(cp), cs1 = *reinterpret_cast<const float4*>(cp + 4);
    const float4 sn0 = *reinterpret_cast<const float4*>(sp), sn1 = *reinterpret_cast<const float4*>(sp + 4);
    const bool has_norm = a.q_gamma != nullptr;
    const uint4 graw = has_norm ? *reinterpret_cast<const uint4*>((it0 < G ? a.q_gamma : a.k_gamma) + sub * 8) : make_uint4(0, 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);

    // ---- this wave's first group of rows ----
    const int end = max(c1 - 1, 0);                              // (beyond the slice its last row again, masked)
    int g0 = c0 + wid * AS_GROUP;
#pragma unroll
    for (int i = 0; i < NI; ++i) kr[i] = at(kc, g0, i, lane, end);
#pragma unroll
    for (int i = 0; i < NI; ++i) vr[i] = at(vc, g0, i, lane, end);
    __builtin_amdgcn_sched_barrier(0);

    auto finish = [&](int it, const float4& lo, const float4& hi, const uint4& gr) {
        float x[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        if (has_norm) {
            float gm[8];
            WTraits<bf16>::decode(gr, gm);
            float ss = 0.f;
#pragma unroll
            for (int j = 0; j < 8; ++j) ss = fmaf(x[j], x[j], ss);
            ss = group_sum<LPR>(ss);
            const float inv = 1.0f / sqrtf(ss / D + a.eps);
            if (it <= G) {
#pragma unroll
                for (int j = 0; j < 8; ++j) x[j] = x[j] * inv * gm[j];
            }
        }
        const float csv[8] = {cs0.x, cs0.y, cs0.z, cs0.w, cs1.x, cs1.y, cs1.z, cs1.w}, snv[8] = {sn0.x, sn0.y, sn0.z, sn0.w, sn1.x, sn1.y, sn1.z, sn1.w};
        float o[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float other = xor_half<LPR>(x[j]);
            o[j] = sub < LPR / 2 ? (x[j] * csv[j] - other * snv[j]) : (x[j] * csv[j] + other * snv[j]);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = it < G ? o[j] * a.scale : it == G ? o[j] : x[j];
        Vec<bf16> v;
        v.from_float(x);
        if (it < G) q_sh[it][sub] = v.raw;
        else if (it < G + 2) {
            kv_sh[it - G][sub] = v.raw;
            if (owns_new) *reinterpret_cast<uint4*>((it == G ? a.kcache : a.vcache) + head_off + (size_t)pos * D + sub * 8) = v.raw;
        }
    };
    finish(ig, x0, x1, graw);
    if (AS_WAVES * IPW < G + 2)                                  // (workgroup-uniform) groups of 15 and 16 at D = 128
        for (int it = ig + AS_WAVES * IPW; it - ig < G + 2; it += AS_WAVES * IPW) {
            const int ic = min(it, G + 1);
            finish(it, *reinterpret_cast<const float4*>(row + item_off(ic) + sub * 8), *reinterpret_cast<const float4*>(row + item_off(ic) + sub * 8 + 4),
                   has_norm ? *reinterpret_cast<const uint4*>((ic < G ? a.q_gamma : a.k_gamma) + sub * 8) : make_uint4(0, 0, 0, 0));
        }
    __syncthreads();
    if (owns_new)
        for (int g = ig; g - ig < G; g += AS_WAVES * IPW) {      // the new token's score per head
            Vec<bf16> qv, kv;
            qv.raw = q_sh[min(g, G - 1)][sub];
            kv.raw = kv_sh[0][sub];
            float qf[8], kf[8], d = 0.f;
            qv.to_float(qf);
            kv.to_float(kf);
#pragma unroll
            for (int j = 0; j < 8; ++j) d = fmaf(qf[j], kf[j], d);
            d = group_sum<LPR>(d);
            if (sub == 0 && g < G) s_new[g] = d;
        }
    uint4 qf[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        const uint4 v = q_sh[min(l15, G - 1)][4 * ks + q4];
        qf[ks] = l15 < G ? v : make_uint4(0, 0, 0, 0);
    }

    // ---- the slice ----
    char* img = as_smem + wid * as_image<D>();
    float m_run = -INFINITY, l_run = 0.f;                        // of head l15
    f32x4_s o[DT];
#pragma unroll
    for (int i = 0; i < DT; ++i) o[i] = f32x4_s{0.f, 0.f, 0.f, 0.f};
    auto order = []() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); __builtin_amdgcn_wave_barrier(); };
    for (; g0 < c1; g0 += AS_WAVES * AS_GROUP) {
        const int next = g0 + AS_WAVES * AS_GROUP;
        int ln = lane;                                           // opaque: the ~40 LDS addresses are formed anew per group instead of living (and spilling) across the loop
        asm volatile("" : "+v"(ln));
        const int lrow = ln / LPR, lch = ln % LPR, l15 = ln & 15, q4 = ln >> 4, tq = l15 >> 2, tp = l15 & 3;
#pragma unroll
        for (int i = 0; i < NI; ++i) *reinterpret_cast<uint4*>(img + as_koff<D>(i * RPI + lrow, lch)) = kr[i];
        if (next < c1) {
#pragma unroll
            for (int i = 0; i < NI; ++i) kr[i] = at(kc, next, i, ln, end);
        }
        order();
        f32x4_s s[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            s[t] = f32x4_s{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                const uint4 ka = *reinterpret_cast<const uint4*>(img + as_koff<D>(16 * t + l15, 4 * ks + q4));
                s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_s, ka), __builtin_bit_cast(bf16x8_s, qf[ks]), s[t], 0, 0, 0);
            }
        }
        order();
#pragma unroll
        for (int i = 0; i < NI; ++i) *reinterpret_cast<uint4*>(img + as_voff<D>(i * RPI + lrow, lch)) = vr[i];
        if (next < c1) {
#pragma unroll
            for (int i = 0; i < NI; ++i) vr[i] = at(vc, next, i, ln, end);
        }
        // rows = positions g0 + 16 t + 4 q4 + r, column = head l15
        float mx = -INFINITY;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                s[t][r] = g0 + 16 * t + 4 * q4 + r < c1 ? s[t][r] : -INFINITY;
                mx = fmaxf(mx, s[t][r]);
            }
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float m_new = fmaxf(m_run, mx), m_use = m_new == -INFINITY ? 0.f : m_new;      // (a NaN is no maximum, but makes its probability NaN)
        const float alpha = m_new == -INFINITY ? 1.f : __expf(m_run - m_new);
        float ls = 0.f;
        uint32_t pk[4];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            float p[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) p[r] = __expf(s[t][r] - m_use);
            pk[2 * t] = pack_bf16x2(p[0], p[1]);
            pk[2 * t + 1] = pack_bf16x2(p[2], p[3]);
            // the sum runs over the rounded probabilities: numerator and denominator see the same weights
            ls += (__uint_as_float(pk[2 * t] << 16) + __uint_as_float(pk[2 * t] & 0xFFFF0000u)) + (__uint_as_float(pk[2 * t + 1] << 16) + __uint_as_float(pk[2 * t + 1] & 0xFFFF0000u));
        }
        l_run = l_run * alpha + ls;                              // this lane's quarter of the sum
        m_run = m_new;
#pragma unroll
        for (int i = 0; i < DT; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) o[i][r] *= alpha;
        order();
        const uint4 pf = make_uint4(pk[0], pk[1], pk[2], pk[3]);
#pragma unroll
        for (int i = 0; i < DT; ++i) {
            typedef __attribute__((address_space(3))) v4s_s* lds_v4;
            const uint2 u0 = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4)(img + as_voff<D>(4 * q4 + tq, 2 * i + (tp >> 1)) + 8 * (tp & 1))));
            const uint2 u1 = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4)(img + as_voff<D>(16 + 4 * q4 + tq, 2 * i + (tp >> 1)) + 8 * (tp & 1))));
            o[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_s, make_uint4(u0.x, u0.y, u1.x, u1.y)), __builtin_bit_cast(bf16x8_s, pf), o[i], 0, 0, 0);
        }
        order();
    }
    l_run += __shfl_xor(l_run, 16, 64);
    l_run += __shfl_xor(l_run, 32, 64);

    // ---- the waves' states and the new token meet in LDS ----
    __syncthreads();                                             // every wave is done with its image
    float* st = reinterpret_cast<float*>(as_smem);               // [wave][head][D + 4]: o, then m, l
    if (l15 < G) {
        float* mine = st + (wid * G + l15) * RS;
        if (q4 == 0) { mine[D] = m_run; mine[D + 1] = l_run; }
#pragma unroll
        for (int i = 0; i < DT; ++i) *reinterpret_cast<float4*>(mine + 16 * i + 4 * q4) = make_float4(o[i][0], o[i][1], o[i][2], o[i][3]);
    }
    __syncthreads();
    for (int e = threadIdx.x; e < G * D; e += 256) {
        const int g = e / D, d = e % D;
        float ms = owns_new ? s_new[g] : -INFINITY;
#pragma unroll
        for (int w = 0; w < AS_WAVES; ++w) ms = fmaxf(ms, st[(w * G + g) * RS + D]);
        float num = 0.f, den = 0.f;
#pragma unroll
        for (int w = 0; w < AS_WAVES; ++w) {
            const float* r = st + (w * G + g) * RS;
            const float wg = r[D] == -INFINITY ? 0.f : __expf(r[D] - ms);
            num = fmaf(wg, r[d], num);
            den = fmaf(wg, r[D + 1], den);
        }
        if (owns_new) {
            const float wg = __expf(s_new[g] - ms);
            num = fmaf(wg, to_f(reinterpret_cast<const bf16*>(kv_sh[1])[d]), num);
            den += wg;
        }
        if constexpr (DIRECT) {
            const float y = den != 0.f ? num / den : 0.f;
            const size_t at = ((size_t)b * a.hq + (size_t)kvh * G) * D + e;
            if (a.attn_direct16) a.attn_direct16[at] = from_f<bf16>(y);
            else a.attn_direct[at] = y;
        } else {
            float* r = rec + (size_t)g * a.nsplit * (D + 2);
            r[2 + d] = num;
            if (d == 0) { r[0] = ms; r[1] = den; }
        }
    }
    tls.end();
}
