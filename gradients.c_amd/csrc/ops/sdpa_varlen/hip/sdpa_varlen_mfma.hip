/*
 * sdpa_varlen forward on the matrix cores (gfx950): packed causal / windowed / prefix attention over
 * cu_seqlens for F16 tensors with head size 64 or 128 (prefill).  Same contract as the scalar kernel in
 * sdpa_varlen.hip (reference src/ops/sdpa_varlen/metal_sdpa_varlen.metal:137-228, mask :30-55).
 *
 * Work split.  A workgroup of 4 wavefronts owns 128 consecutive query rows of one segment and one query
 * head; a wavefront owns 32 of them.  Keys advance in blocks of 64, staged in LDS (K and V, two stages,
 * global -> LDS loads that bypass the registers) and shared by the four wavefronts.
 *
 * Transposed formulation.  Both products are computed transposed so that a query row lives in ONE lane
 * (column l%32 of every v_mfma_f32_32x32x16_f16 result) and its keys / channels in that lane's registers:
 *     S^T = K   Q^T    (A = K rows from LDS, B = Q kept in registers for the whole kernel)
 *     O^T = V^T P^T    (A = V^T gathered by ds_read_b64_tr_b16, B = P^T = the S^T registers, rounded to F16)
 * Row maxima and sums are then in-lane reductions plus one exchange with lane l^32, the rescale of O by
 * exp2(m_old - m_new) is a per-lane scalar, and P never moves between lanes: result register 4a+r of S^T
 * is key 8a + 4*(l/32) + r of a 32-key tile, and eight consecutive registers are exactly the eight k-slots
 * of lane l for one 16-key step of the second product, provided V^T supplies the same keys in the same
 * slots - which the transposing LDS read can do for any choice of rows.
 *
 * Softmax in the exp2 domain: s = (q.k) * scale * log2(e), F32 throughout; probabilities are rounded to F16
 * only as the operand of the second product, the row sum accumulates the unrounded values.  The scaling rides in
 * the multiply-add in front of the exp2, and the running maximum of a row moves (O and the row sum rescaled) only
 * when a block raises it by more than 8 binary orders: the result does not depend on the reference point.
 *
 * What it takes (32 prompts of 64 to 2048 rows, 16 heads of 128): 355 us, 410 before the key rows' addresses, the clearing of V
 * rows and the zeroing of score registers left the loop (buffer descriptors that follow the block and end with the segment;
 * fragment addresses computed once; the first product over a zero accumulator), before masks became plain comparisons with the
 * row's limits (branches per key before: 16 prompts of 20 to 400 rows through a window of 256, 8 heads of 64, 33.7 -> 15.1 us),
 * and before the longest prompts came first.  Vector and matrix instructions are each busy a third of the time; wavefronts wait
 * at the block's barrier and for each other.
 *
 * LDS layouts (16-byte chunks, CPR = D/8 per row).  K: chunk c of key row r at position c ^ (r & 15)
 * (D = 128) or c ^ ((r >> 1) & 7) (D = 64): the 16 lanes of a fragment read hit 16 different bank groups.
 * V: chunk c of key row r at c ^ ((r & 3) << 2) (D = 128) or c ^ (((r >> 1) & 1) << 2) (D = 64): the four
 * key rows of a transposing read cover all banks.
 */
#include "../../_shared/hip_row_blocks.h"
#include <type_traits>

#define GD_VL_NEG_INF (-__builtin_inff())

struct gd_hip_sdpa_varlen_params {
    uint32_t n_rows, batch, hq, hkv, dh;
    uint32_t causal, window, prefix_len, max_seqlen;
    float scale;
    uint32_t kv_tmax; /* 0: k and v are packed like q; otherwise caches [batch, kv_tmax, hkv, dh], token t of
                         segment b in cache row t of sequence b */
};

typedef int gd_vl_int4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) unsigned char gd_vl_lds;

/* 16 bytes per lane from global memory straight into LDS (lane l's data lands at lds + IMM + 16 l); lanes behind the
 * descriptor's range get zeros.  Assembly, because the compiler would otherwise wait for every outstanding load before
 * each LDS read; the kernel places its own s_waitcnt vmcnt. */
template <int IMM>
__device__ __forceinline__ void gd_vl_load_lds16(gd_vl_int4 descriptor, uint32_t lane_bytes, uint32_t lds)
{
    asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %3, 0 offen lds"
                 :
                 : "s"(lds), "n"(IMM), "v"(lane_bytes), "s"(descriptor)
                 : "memory", "scc");
}

template <int D>
__global__ void __launch_bounds__(256, 2)
gd_sdpa_varlen_mfma_kernel(const gd_half *__restrict__ q, const gd_half *__restrict__ k, const gd_half *__restrict__ v,
                           const int32_t *__restrict__ cu, gd_half *__restrict__ out, gd_hip_sdpa_varlen_params p)
{
    constexpr uint32_t BQ = 128u, BKEYS = 64u;
    constexpr uint32_t CPR = D / 8u;            /* 16-byte chunks per row */
    constexpr uint32_t RPL = 64u / CPR;         /* key rows per wavefront load */
    constexpr int LOADS = (int)(BKEYS / RPL / 4u); /* wavefront loads per operand, key block and wavefront */
    constexpr uint32_t TILE_CHUNKS = BKEYS * CPR; /* one K or V block */
    constexpr int KSTEPS = D / 16, DTILES = D / 32;
    typedef short gd_short4 __attribute__((ext_vector_type(4)));
    extern __shared__ __align__(16) unsigned char gd_vl_smem[]; /* [2 stages][K block, V block] */

    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t lq = lane & 31u, h = lane >> 5;
    const uint32_t hq = blockIdx.x % p.hq, pair = blockIdx.x / p.hq;
    const uint32_t hkv = hq / (p.hq / p.hkv);

    if (cu[0] < 0) return;
    gd_row_block at;
    if (!gd_find_row_block(cu, p.batch, BQ, pair, &at) || at.end > (int)p.n_rows) return;
    const uint32_t b = at.seq;
    const int start = at.start, end = at.end;
    const int T_len = end - start;
    if (p.kv_tmax != 0u && (uint32_t)T_len > p.kv_tmax) return; /* a segment its cache cannot hold: out stays */
    /* row of K and V that holds the segment's first key */
    const uint32_t kv_first = p.kv_tmax != 0u ? b * p.kv_tmax : (uint32_t)start;
    const int i0 = (int)(at.block * BQ);
    const int causal = (int)p.causal, window = (int)p.window, prefix = (int)p.prefix_len;

    /* key blocks this workgroup walks */
    const int i_last = min(i0 + (int)BQ, T_len) - 1;
    int kend = T_len, kbeg = 0;
    if (causal) {
        kend = min(T_len, i_last + 1);
        if (prefix > 0 && i0 < prefix) kend = max(kend, min(T_len, prefix));
    }
    if (window > 0 && prefix == 0) kbeg = max(0, i0 - window + 1) & ~63;

    /* this lane's query row */
    const int wi0 = i0 + (int)wave * 32;          /* first row of the wavefront */
    const int i = wi0 + (int)lq;
    const bool row_live = i < T_len;
    const size_t q_elem = ((size_t)(start + min(i, T_len - 1)) * p.hq + hq) * D;
    gd_half8 qf[KSTEPS];
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
        qf[ks] = (gd_half8)(gd_half)0.f;
        if (row_live) qf[ks] = *reinterpret_cast<const gd_half8 *>(q + q_elem + 16 * ks + 8 * h);
    }

    /* Staging.  A load of this wavefront fills RPL key rows; lane offsets do not depend on the block, whose rows the
     * descriptor's base and range follow: rows behind the segment's end (another segment's, or a cache's free ones) arrive
     * as zeros, so that probability 0 times their values is 0. */
    gd_vl_lds *const smem = (gd_vl_lds *)gd_vl_smem;
    const uint32_t row_pitch = p.hkv * D * 2u; /* bytes between consecutive key rows */
    const uint32_t lds_wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)(uintptr_t)smem + wave * (uint32_t)LOADS * 1024u));
    uint32_t off_k[LOADS], off_v[LOADS];
#pragma unroll
    for (int t = 0; t < LOADS; ++t) {
        const uint32_t r = (wave * (uint32_t)LOADS + (uint32_t)t) * RPL + lane / CPR, pos = lane % CPR;
        off_k[t] = r * row_pitch + (pos ^ (D == 128 ? (r & 15u) : ((r >> 1) & 7u))) * 16u;
        off_v[t] = r * row_pitch + (pos ^ (D == 128 ? ((r & 3u) << 2) : (((r >> 1) & 1u) << 2))) * 16u;
    }
    const uint32_t segment = (uint32_t)__builtin_amdgcn_readfirstlane((int)kv_first);
    const uint32_t keys = (uint32_t)__builtin_amdgcn_readfirstlane(T_len);
    /* the key block jb of K or V (part 0, 1) into a stage; jb < keys */
    auto request = [&](auto part, int jb, uint32_t stage) __attribute__((always_inline)) {
        constexpr int V = decltype(part)::value, AT = V * (int)TILE_CHUNKS * 16;
        const uint64_t first = (uint64_t)(V ? v : k) + (uint64_t)(segment + (uint32_t)jb) * row_pitch + hkv * D * 2u;
        const uint32_t range = min(keys - (uint32_t)jb - 1u, BKEYS - 1u) * row_pitch + D * 2u;
        gd_vl_int4 of;
        of[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)first);
        of[1] = __builtin_amdgcn_readfirstlane((int)(uint32_t)(first >> 32));
        of[2] = __builtin_amdgcn_readfirstlane((int)range);
        of[3] = 0x00020000; /* untyped, no swizzle */
        const uint32_t to = lds_wave + stage * (2u * TILE_CHUNKS * 16u);
        const uint32_t (&off)[LOADS] = V ? off_v : off_k;
        gd_vl_load_lds16<AT>(of, off[0], to);
        gd_vl_load_lds16<AT + 1024>(of, off[1], to);
        if constexpr (LOADS == 4) {
            gd_vl_load_lds16<AT + 2048>(of, off[LOADS - 2], to);
            gd_vl_load_lds16<AT + 3072>(of, off[LOADS - 1], to);
        }
    };
    using gd_k = std::integral_constant<int, 0>;
    using gd_v = std::integral_constant<int, 1>;
    static_assert(LOADS == 2 || LOADS == 4, "the loads above");

    gd_float16 o[DTILES];
#pragma unroll
    for (int t = 0; t < DTILES; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[t][e] = 0.f;
    float m = GD_VL_NEG_INF, l = 0.f;
    const float scale2 = p.scale * 1.4426950408889634f;
    const bool plain_causal = causal != 0 && window == 0 && prefix == 0;
    /* visible keys of this lane's row: up to jmax, but for jfrom .. jgone */
    int jmax = T_len - 1;
    if (causal) jmax = min(jmax, prefix > 0 && i < prefix ? prefix - 1 : i);
    const int jgone = window > 0 && (prefix == 0 || i >= prefix) ? i - window : -1, jfrom = prefix;

    /* Fragment addresses in the first stage; what a step of K or of the channels changes is a xor with a constant, key rows
     * and the V block are immediate offsets.
     * K: key row lq (+ 32 t), chunk 2 ks + h.  V, transposing reads: group g = lane / 16 -> channel block 16 (g & 1), key
     * half g / 2 == h; lane q + 4 e of a group addresses key row e (+ 4 h + 16 ts, + 8 the second), channels 4 q .. + 3. */
    const uint32_t tr_q = lane & 3u, tr_e = (lane >> 2) & 3u, tr_g1 = (lane >> 4) & 1u;
    const uint32_t v_row = 4u * h + tr_e; /* the swizzle of rows 8 and 16 ts behind it is the same */
    uint32_t at_k[KSTEPS], at_v[DTILES];
#pragma unroll
    for (uint32_t ks = 0; ks < (uint32_t)KSTEPS; ++ks)
        at_k[ks] = (lq * CPR + ((2u * ks + h) ^ (D == 128 ? (lq & 15u) : ((lq >> 1) & 7u)))) * 16u;
#pragma unroll
    for (uint32_t dt = 0; dt < (uint32_t)DTILES; ++dt)
        at_v[dt] = (TILE_CHUNKS + v_row * CPR + ((4u * dt + 2u * tr_g1 + (tr_q >> 1)) ^ (D == 128 ? (tr_e << 2) : (((v_row >> 1) & 1u) << 2)))) * 16u +
                   (tr_q & 1u) * 8u;

    /* The scores of a block are computed while the block in front of it is exponentiated: matrix and vector instructions of
     * one wavefront side by side.  So K runs a block ahead of V. */
    auto key = [&](uint32_t stage, int n) __attribute__((always_inline)) { /* fragment n = t * KSTEPS + ks */
        return *(__attribute__((address_space(3))) gd_half8 *)(smem + stage * (2u * TILE_CHUNKS * 16u) + at_k[n % KSTEPS] +
                                                               32u * (uint32_t)(n / KSTEPS) * CPR * 16u);
    };
    auto value = [&](uint32_t stage, int n) __attribute__((always_inline)) {
        gd_vl_lds *const at = smem + stage * (2u * TILE_CHUNKS * 16u) + at_v[n % DTILES] + 16u * (uint32_t)(n / DTILES) * CPR * 16u;
        union { gd_short4 s[2]; gd_half8 hv; } u;
        u.s[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) gd_short4 *)at);
        u.s[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) gd_short4 *)(at + 8u * CPR * 16u));
        return u.hv;
    };
    gd_float16 st0[2], st1[2];
    request(gd_k{}, kbeg, 0u);
    request(gd_v{}, kbeg, 0u);
    if (kbeg + (int)BKEYS < kend) request(gd_k{}, kbeg + (int)BKEYS, 1u);
    __builtin_amdgcn_s_waitcnt(0x0F70); /* vmcnt(0) */
    __syncthreads();
#pragma unroll
    for (int n = 0; n < 2 * KSTEPS; ++n)
        st0[n / KSTEPS] = __builtin_amdgcn_mfma_f32_32x32x16_f16(key(0u, n), qf[n % KSTEPS], n % KSTEPS == 0 ? (gd_float16)(0.f) : st0[n / KSTEPS], 0, 0, 0);
    /* block jb, whose K and V lie in `stage`: its scores st, the next block's go to `next` */
    auto walk = [&](gd_float16 (&st)[2], gd_float16 (&next)[2], int jb, auto stage_tag) __attribute__((always_inline)) {
        constexpr uint32_t stage = decltype(stage_tag)::value;
        __builtin_amdgcn_s_waitcnt(0x0F70); /* vmcnt(0): this wavefront's share of V of block jb and of the next K is in LDS */
        __syncthreads();                    /* everyone's share is; K of block jb and V of the one in front are no longer read */
        if (jb + (int)BKEYS < kend) request(gd_v{}, jb + (int)BKEYS, stage ^ 1u);
        if (jb + 2 * (int)BKEYS < kend) request(gd_k{}, jb + 2 * (int)BKEYS, stage);
        /* a causal wavefront whose rows all precede the block has nothing to add, nor from the blocks behind it */
        const bool wave_needs = !causal || jb <= wi0 + 31 || (prefix > 0 && jb < prefix);
        if (!wave_needs) return;

        /* scale, mask, block maximum.  The scores stay unscaled in their registers: scale2 > 0, so the maximum of the
         * raw values is the raw value of the maximum, and the scaling rides in the multiply-add in front of the exp2. */
        const bool full = jb + (int)BKEYS <= T_len &&
                          (causal ? (prefix == 0 && jb + 63 <= wi0 && (window == 0 || wi0 + 31 - jb < window))
                                  : (window == 0));
        float mraw = GD_VL_NEG_INF;
        if (!full && plain_causal) { /* no window, no prefix: one comparison against min(i, T_len - 1) */
            const int behind = jmax - jb - 4 * (int)h;
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int e = 0; e < 16; ++e) st[t][e] = 32 * t + 8 * (e >> 2) + (e & 3) > behind ? GD_VL_NEG_INF : st[t][e];
        } else if (!full) {
#pragma unroll
            for (int t = 0; t < 2; ++t) {
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int j = jb + 32 * t + 8 * (e >> 2) + 4 * (int)h + (e & 3);
                    const bool hidden = (j > jmax) | ((j <= jgone) & (j >= jfrom));
                    st[t][e] = hidden ? GD_VL_NEG_INF : st[t][e];
                }
            }
        }
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int e = 0; e < 16; ++e) mraw = fmaxf(mraw, st[t][e]);
        float mloc = mraw * scale2; /* -inf stays -inf */
        mloc = fmaxf(mloc, __shfl_xor(mloc, 32, 64));
        /* The running maximum is only a reference point: the result does not depend on it as long as nothing
         * overflows.  It moves (and O and the row sum are rescaled) only when some row of the wavefront has found a
         * score more than 8 binary orders above its reference, or has none yet; until then the probabilities of a
         * block may reach 2^8, which F16 holds with its full precision, and 64 multiplications per block are saved. */
        const bool moves = mloc > m + 8.f || (m == GD_VL_NEG_INF && mloc != GD_VL_NEG_INF);
        if (__builtin_amdgcn_ballot_w64(moves) != 0ull) {
            const float mnew = fmaxf(m, mloc);
            const float msafe_new = mnew == GD_VL_NEG_INF ? 0.f : mnew;
            const float corr = __builtin_amdgcn_exp2f(m - msafe_new); /* m = -inf -> 0 */
            l *= corr;
            m = mnew;
#pragma unroll
            for (int t = 0; t < DTILES; ++t)
#pragma unroll
                for (int e = 0; e < 16; ++e) o[t][e] *= corr;
        }
        const float msafe = m == GD_VL_NEG_INF ? 0.f : m;
        /* probabilities of this block beside the scores of the next (of stale keys behind the last block: not used) */
        constexpr int NK = 2 * KSTEPS, PER = 32 / NK, AHEAD = 4;
        float psum = 0.f;
        gd_half8 pf[4], kf[AHEAD], vf[AHEAD];
#pragma unroll
        for (int n = 0; n < AHEAD; ++n) kf[n] = key(stage ^ 1u, n);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int n = 0; n < NK; ++n) {
            next[n / KSTEPS] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[n % AHEAD], qf[n % KSTEPS], n % KSTEPS == 0 ? (gd_float16)(0.f) : next[n / KSTEPS], 0, 0, 0);
            if (n + AHEAD < NK) kf[n % AHEAD] = key(stage ^ 1u, n + AHEAD);
            else vf[n + AHEAD - NK] = value(stage, n + AHEAD - NK);
#pragma unroll
            for (int x = n * PER; x < (n + 1) * PER; ++x) {
                const int t = x / 16, e = x % 16;
                const float pe = __builtin_amdgcn_exp2f(fmaf(st[t][e], scale2, -msafe));
                psum += pe;
                pf[2 * t + (e >> 3)][e & 7] = (gd_half)pe;
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        l += psum;

        /* O^T += V^T P^T: fragment n = channel tile n % DTILES of 16-key step n / DTILES, four of them on their way */
        constexpr int NV = 4 * DTILES;
#pragma unroll
        for (int n = 0; n < NV; ++n) {
            o[n % DTILES] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[n % AHEAD], pf[n / DTILES], o[n % DTILES], 0, 0, 0);
            if (n + AHEAD < NV) vf[n % AHEAD] = value(stage, n + AHEAD);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    for (int jb = kbeg; jb < kend;) {
        walk(st0, st1, jb, std::integral_constant<uint32_t, 0>{});
        jb += (int)BKEYS;
        if (jb >= kend) break;
        walk(st1, st0, jb, std::integral_constant<uint32_t, 1>{});
        jb += (int)BKEYS;
    }

    /* normalise, then through LDS so that rows leave with 16-byte stores */
    l += __shfl_xor(l, 32, 64);
    const bool zero_row = p.max_seqlen > 0u && i >= (int)p.max_seqlen;
    const float inv = (l > 0.f && !zero_row) ? 1.f / l : 0.f;
    __syncthreads(); /* all fragment reads of the last block are done */
    gd_half *sO = reinterpret_cast<gd_half *>(gd_vl_smem) + (size_t)wave * 32u * D;
#pragma unroll
    for (int dt = 0; dt < DTILES; ++dt) {
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            gd_half4 hv;
#pragma unroll
            for (int r = 0; r < 4; ++r) hv[r] = (gd_half)(o[dt][4 * a + r] * inv);
            *reinterpret_cast<gd_half4 *>(sO + lq * D + 32 * dt + 8 * a + 4 * h) = hv;
        }
    }
    __syncthreads();
    for (uint32_t c = lane; c < 32u * CPR; c += 64u) {
        const uint32_t r = c / CPR, cc = c % CPR;
        const int ri = wi0 + (int)r;
        if (ri < T_len)
            *reinterpret_cast<gd_half8 *>(out + ((size_t)(start + ri) * p.hq + hq) * D + cc * 8u) =
                *reinterpret_cast<const gd_half8 *>(sO + r * D + cc * 8u);
    }
}

/* F16, head size 64 or 128, every row pitch a multiple of 16 bytes, tensors below 4 GiB.  The grid has one
 * workgroup per (128-row block of a segment, query head); blocks past the last segment exit at once. */
extern "C" int gd_hip_launch_sdpa_varlen_mfma(hipStream_t stream, const void *q, const void *k, const void *v,
                                              const int32_t *cu, void *out, uint32_t n_rows, uint32_t batch,
                                              uint32_t hq, uint32_t hkv, uint32_t dh, uint32_t causal, uint32_t window,
                                              uint32_t prefix_len, uint32_t max_seqlen, float scale,
                                              uint32_t kv_tmax)
{
    gd_hip_sdpa_varlen_params p = {n_rows, batch, hq, hkv, dh, causal, window, prefix_len, max_seqlen, scale, kv_tmax};
    const uint64_t pairs = (uint64_t)(n_rows + 127u) / 128u + batch; /* upper bound of sum ceil(len_b / 128) */
    const uint64_t blocks = pairs * hq;
    if (n_rows == 0u || blocks == 0u) return (int)hipSuccess;
    if (blocks > 0x7fffffffull) return (int)hipErrorInvalidValue;
    if (dh == 128u) {
        const size_t lds = 2u * 2u * 64u * 16u * 16u;
        static bool configured = false;
        if (!configured) {
            const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(gd_sdpa_varlen_mfma_kernel<128>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            if (e != hipSuccess) return (int)e;
            configured = true;
        }
        gd_sdpa_varlen_mfma_kernel<128><<<(unsigned)blocks, 256, lds, stream>>>(
            (const gd_half *)q, (const gd_half *)k, (const gd_half *)v, cu, (gd_half *)out, p);
    } else {
        const size_t lds = 2u * 2u * 64u * 8u * 16u;
        gd_sdpa_varlen_mfma_kernel<64><<<(unsigned)blocks, 256, lds, stream>>>(
            (const gd_half *)q, (const gd_half *)k, (const gd_half *)v, cu, (gd_half *)out, p);
    }
    return (int)hipGetLastError();
}
