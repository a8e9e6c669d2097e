/*
 * Instantiations and launcher of gd_linear_wide_kernel (linear_wide_kernel.h): the few-row projections of the wide
 * decoders.  A translation unit of its own, like linear_lds.hip, so that the code object of linear.hip stays as it
 * is laid out without it.
 */
#include "linear_wide_kernel.h"

template <int NT, int MT, int PMAX, int PRO, int EPI>
static void launch_wide(hipStream_t stream, const void *x, const void *w, const void *bias, const void *residual,
                        const void *norm_w, void *y, const gd_hip_linear_params &p, const gd_hip_rope_epilogue &rope)
{
    constexpr bool PAIRED = EPI != GD_WIDE_EPI_PLAIN;
    const uint32_t cols = PAIRED ? 8u * NT : 16u * NT; /* output (first-of-pair) columns per workgroup */
    const uint32_t outs = EPI == GD_WIDE_EPI_ROPE ? p.N / 2u : (EPI == GD_WIDE_EPI_SWIGLU ? p.swiglu_cols : p.N);
    const uint32_t n_tiles = outs / cols;
    dim3 grid(n_tiles, (p.M + 16u * MT - 1u) / (16u * MT));
    gd_linear_wide_kernel<NT, MT, PMAX, 8, PRO, EPI><<<grid, 512, 0, stream>>>(
        (const gd_elem *)x, (const gd_elem *)w, (const gd_elem *)bias, (const gd_elem *)residual,
        (const gd_elem *)norm_w, (gd_elem *)y, p, n_tiles, rope);
}

/* 8 columns per workgroup (narrow outputs, one row tile): see gd_linear_wide_half_kernel */
template <int QMAX>
static void launch_wide_half(hipStream_t stream, const void *x, const void *w, const void *bias, const void *residual,
                             void *y, const gd_hip_linear_params &p)
{
    const uint32_t n_tiles = p.N / 8u;
    dim3 grid(n_tiles, (p.M + 15u) / 16u);
    gd_linear_wide_half_kernel<QMAX, 8><<<grid, 512, 0, stream>>>(
        (const gd_elem *)x, (const gd_elem *)w, (const gd_elem *)bias, (const gd_elem *)residual, (gd_elem *)y, p, n_tiles);
}

/* persistent form: at most 8 tiles per workgroup, one workgroup per compute unit; outputs in tiles of 16 * NT columns (paired
 * epilogues: 8 * NT), the last one perhaps not full.  F16: K = 2048 behind an rms_norm.  false: nothing launched, because fewer
 * than min_tiles workgroups would stream */
template <int NT, int MT, int PMAX, int EPI, int PRO>
static bool launch_persistent(hipStream_t stream, const void *x, const void *w, const void *bias, const void *residual,
                              const void *norm_w, void *y, const gd_hip_linear_params &p, const gd_hip_rope_epilogue &rope,
                              uint32_t units, bool narrow, uint32_t min_tiles)
{
    constexpr bool PAIRED = EPI != GD_WIDE_EPI_PLAIN;
    /* as deep as LDS allows next to the sums of the wavefronts (NT x MT x 8 KB): 8 x RING x 2 KB; an eighth group for
     * the two-tile forms changed nothing (12.5 against 12.2 us at 16 x 2048 -> 6144) */
    constexpr int RING = NT * MT <= 4 ? 7 : 5;
    const uint32_t cols = PAIRED ? 8u * NT : 16u * NT;
    const uint32_t outs = EPI == GD_WIDE_EPI_ROPE ? p.N / 2u : (EPI == GD_WIDE_EPI_SWIGLU ? p.swiglu_cols : p.N);
    uint32_t n_tiles = (outs + cols - 1u) / cols, tile_w = cols;
    /* fewer full tiles than compute units (5632 gated outputs: 176 tiles of 32): narrower tiles, one per unit, so
     * that every unit streams its share of the weights (22 columns each; the 3072 rotation pairs of a 6144-row qkv
     * weight: 12 pairs each).  Narrow rope tiles straddle heads: only when half the head size is a power of two. */
    const uint32_t hd2 = p.rope_head_dim / 2u;
    const bool may_straddle = EPI != GD_WIDE_EPI_ROPE || (hd2 != 0u && (hd2 & (hd2 - 1u)) == 0u);
    if (may_straddle && n_tiles < units && narrow && 2u * ((outs + units - 1u) / units) > cols) {
        tile_w = (outs + units - 1u) / units; /* more than half of a tile's columns stay in use */
        n_tiles = (outs + tile_w - 1u) / tile_w;
    }
    if (n_tiles < min_tiles) return false;
    uint32_t groups = n_tiles < units ? n_tiles : units;
    if ((n_tiles + groups - 1u) / groups > 8u) groups = (n_tiles + 7u) / 8u;
    dim3 grid(groups, (p.M + 16u * MT - 1u) / (16u * MT));
    gd_linear_wide_persistent_kernel<NT, MT, PMAX, RING, EPI, 8, PRO><<<grid, 512, 0, stream>>>(
        (const gd_elem *)x, (const gd_elem *)w, (const gd_elem *)bias, (const gd_elem *)residual,
        (const gd_elem *)norm_w, (gd_elem *)y, p, n_tiles, tile_w, rope);
    return true;
}

#if GD_LINEAR_IS_BF16
/* BF16: the widest column tiles that leave at most a quarter of the compute units without one (with fewer workgroups the
 * 16-column form streams faster).  Four row tiles keep 32 columns (their sums would not fit beside the ring), and K = 4096 two
 * row tiles (registers).  Against the 16-column form, which reads x (as many bytes as its weights) for every 16 columns and the
 * weights for every 16 rows, and against the stream kernel for gated outputs, weights from HBM (us; 4, 16, 32, 64 rows):
 *   1024 -> 32768 F32 results  15.5, 15.9, 18.1, 22.2 (24.7, 29.1, 53.1, 99.9): 4.3 to 3.0 TB/s
 *   2048 -> 32768 F32 results  30.1, 29.6, 31.8, 37.2 (37.1, 38.6, 67.3, 121): 4.5 to 3.6 TB/s
 *   1024 -> 2816 gated         5.1, 5.1, 6.1, 8.7 (5.9, 6.4, 8.6, 14.3);  2048 -> 5632 gated 12.2, 12.8, 14.9, 21.0 (15.9, 16.5, 26.3, 37.1)
 *   1024 -> 4384               4.6, 4.8, 5.8, 8.3 (6.6, 7.7, 11.0, 17.5);  4096 -> 8448 17.5, 19.1, 22.8, 41.0 (24.1, 31.0, 48.3, 82.8)
 * and for the K between the powers of two (us; 1, 16, 32, 64 rows):
 *   1536 -> 32768 F32 results  21.7, 22.4, 24.6, 29.3 (26.8, 34.3, 60.2, 112);  3072 -> 32768 41.7, 40.8, 44.3, 77.2 (48.7, 73.5, 135, 257)
 *   1536 -> 6144               6.2, 7.1, 8.3, 11.6 (7.6, 9.6, 13.0, 22.6);  2560 -> 6144 8.6, 10.0, 12.6, 21.0 (12.5, 18.6, 26.1, 48.7)
 *   512 -> 8448 gated          7.5, 8.1, 9.4, 11.4 (8.4, 9.0, 11.2, 15.6);  1536 -> 4224 gated 8.4, 9.3, 10.9, 15.8 (11.3, 12.5, 20.8, 30.1)
 *   3072 -> 8448 gated         29.0, 30.5, 34.6, 58.7 (37.7, 41.0, 55.5, 85.8);  3584 -> 3072 gated 11.3, 12.8, 16.3, 28.1 (12.8, 15.1, 22.9, 38.9) */
template <int PMAX, int EPI>
static bool launch_persistent_rows(hipStream_t stream, const void *x, const void *w, const void *bias, void *y,
                                   const gd_hip_linear_params &p, const gd_hip_rope_epilogue &rope, uint32_t units)
{
    const uint32_t least = units - units / 4u;
#define GD_P(NT, MT) launch_persistent<NT, MT, PMAX, EPI, GD_HIP_PRO_NONE>(stream, x, w, bias, nullptr, nullptr, y, p, rope, units, true, least)
    if (p.M <= 16u) return GD_P(4, 1) || GD_P(2, 1);
    if constexpr (PMAX <= 4) {
        if (p.M > 32u) return GD_P(2, 4);
    }
    return GD_P(4, 2) || GD_P(2, 2);
#undef GD_P
}
#endif

/* Returns the form (GD_HIP_LINEAR_WIDE_*) that took the launch (hipGetLastError() then tells how it went), 0 when this
 * kernel family does not cover the call and the caller goes on to the stream kernel.  Covered: [N,K] weights of at least
 * min_bytes and below 2^29 elements (byte offsets of both sections of a paired weight in 31 bits; plain weights beyond that,
 * 131,072 x 4096, take the stream kernel) whose K is a multiple of 64, fewer than 128 rows, and
 *   BF16, K = 512 to 4096 in steps of 512, column tiles for three quarters of the compute units: plain and gated in the
 *                     persistent form (launch_persistent_rows);
 *   plain epilogue:   no prologue, 16 columns per workgroup (8 where that leaves compute units without one), K that splits
 *                     over the eight wavefronts into at most 12 pairs of steps each; F16 behind an rms_norm, at most 4
 *                     pairs, 64 columns per workgroup;
 *   swiglu epilogue:  F16 behind an rms_norm, 32 (tiles == 2) or 64 weight rows per workgroup;
 *   rope epilogue:    F16 behind an rms_norm, 32 weight rows per workgroup (head size a multiple of 32). */
extern "C" int GD_LINEAR_FN(gd_hip_try_launch_linear_wide)(hipStream_t stream, const void *x, const void *w, const void *bias,
                                             const void *residual, const void *norm_w, void *y,
                                             const gd_hip_linear_params *params, const gd_hip_rope_epilogue *rope_epilogue,
                                             uint64_t min_bytes, uint32_t tiles, uint32_t units)
{
    const gd_hip_rope_epilogue no_rope = {nullptr, nullptr, nullptr, nullptr, nullptr};
    const gd_hip_rope_epilogue &rope = rope_epilogue != nullptr ? *rope_epilogue : no_rope;
    const gd_hip_linear_params &p = *params;
    if (!p.w_is_nk || p.M == 0u || p.M >= 128u || p.K == 0u || (p.K % 64u) != 0u ||
        (uint64_t)p.N * p.K * 2u < min_bytes || (uint64_t)p.N * p.ldw * 4u >= 0x7fffffffull ||
        (uint64_t)p.M * p.ldx * 2u >= 0x7fffffffull)
        return 0;
    const uint32_t ppw = (p.K / 64u + 7u) / 8u; /* pairs of steps per wavefront */
    const int epi = p.rope_head_dim != 0u ? GD_WIDE_EPI_ROPE : (p.swiglu_cols != 0u ? GD_WIDE_EPI_SWIGLU : GD_WIDE_EPI_PLAIN);
    const uint32_t mt = p.M <= 16u ? 1u : (p.M <= 32u ? 2u : 4u);
#if GD_LINEAR_IS_BF16
    /* K that the eight wavefronts share in whole pairs of steps, up to the pairs whose activations fit a lane's registers: the
     * persistent form; other K and narrower outputs go on */
    if (tiles != 1u && p.prologue == GD_HIP_PRO_NONE && epi != GD_WIDE_EPI_ROPE && (p.K % 512u) == 0u) {
#define GD_R(PMAX)                                                                                                           \
    case PMAX:                                                                                                              \
        if (epi == GD_WIDE_EPI_PLAIN ? launch_persistent_rows<PMAX, GD_WIDE_EPI_PLAIN>(stream, x, w, bias, y, p, rope, units) \
                                     : launch_persistent_rows<PMAX, GD_WIDE_EPI_SWIGLU>(stream, x, w, bias, y, p, rope, units)) \
            return GD_HIP_LINEAR_WIDE_PERSISTENT;                                                                           \
        break
        switch (p.K / 512u) {
            GD_R(1); GD_R(2); GD_R(3); GD_R(4); GD_R(5); GD_R(6); GD_R(7); GD_R(8);
        }
#undef GD_R
    }
#endif
    const bool persistent = tiles != 1u; /* "linear_tiles" = 1 asks for the one-tile-per-workgroup form (for comparison) */
#define GD_W(NT, MT, PMAX, PRO, EPI) \
    do { launch_wide<NT, MT, PMAX, PRO, EPI>(stream, x, w, bias, residual, norm_w, y, p, rope); return GD_HIP_LINEAR_WIDE_TILE; } while (0)
#define GD_W_MT(NT, PMAX, PRO, EPI) \
    do { if (mt == 1u) GD_W(NT, 1, PMAX, PRO, EPI); if (mt == 2u) GD_W(NT, 2, PMAX, PRO, EPI); GD_W(NT, 4, PMAX, PRO, EPI); } while (0)
    if (p.prologue == GD_HIP_PRO_NONE && epi == GD_WIDE_EPI_PLAIN && (p.N % 16u) == 0u) {
        /* 16 columns per workgroup: these are the narrow outputs (N = d_model), where further row tiles are worth
         * more as workgroups of their own (16 x 2048 x 2048 and 32 x ...: 6.0 us with one row tile per workgroup,
         * 8.2 us with both in one; the second reader of a weight line finds it in L2) */
        /* up to 16 rows and fewer 16-column tiles than compute units: 8 columns per workgroup, so that every unit
         * streams (16 x 5632 -> 2048: 256 workgroups instead of 128) */
        if (p.M <= 16u && p.N / 16u < units && tiles != 1u && (p.K % 128u) == 0u && (p.N % 8u) == 0u) {
            const uint32_t qpw = (p.K / 128u + 7u) / 8u; /* pieces of 128 per wavefront */
            if (qpw <= 2u) { launch_wide_half<2>(stream, x, w, bias, residual, y, p); return GD_HIP_LINEAR_WIDE_HALF; }
            if (qpw <= 6u) { launch_wide_half<6>(stream, x, w, bias, residual, y, p); return GD_HIP_LINEAR_WIDE_HALF; }
#if GD_LINEAR_IS_BF16
            /* (8448 -> 2048 at 4 and 16 rows: 12.7 and 17.0 us, the stream kernel's four wavefronts 14.7 and 18.3; what is left is the
             * activation matrix, which every 8 columns read whole) */
            if (qpw <= 12u) { launch_wide_half<12>(stream, x, w, bias, residual, y, p); return GD_HIP_LINEAR_WIDE_HALF; }
#endif
        }
        if (ppw <= 4u) GD_W(1, 1, 4, GD_HIP_PRO_NONE, GD_WIDE_EPI_PLAIN);
        if (ppw <= 12u) GD_W(1, 1, 12, GD_HIP_PRO_NONE, GD_WIDE_EPI_PLAIN);
        return 0;
    }
#if GD_LINEAR_IS_BF16
    (void)persistent;
    (void)mt;
#else
    if (p.prologue != GD_HIP_PRO_RMS_NORM || ppw > 4u) return 0;
    /* K = 2048: the persistent form, where its LDS holds the sums of MT x NT tiles next to the ring */
#define GD_P(NT, MT, EPI) \
    do { launch_persistent<NT, MT, 4, EPI, GD_HIP_PRO_RMS_NORM>(stream, x, w, bias, residual, norm_w, y, p, rope, units, tiles != 4u, 0u); return GD_HIP_LINEAR_WIDE_PERSISTENT; } while (0)
    if (p.K == 2048u && persistent) {
        if (epi == GD_WIDE_EPI_PLAIN && (p.N % 64u) == 0u && mt <= 2u) {
            if (mt == 1u) GD_P(4, 1, GD_WIDE_EPI_PLAIN);
            GD_P(4, 2, GD_WIDE_EPI_PLAIN);
        }
        /* four row tiles: the sums of 4 x 4 tiles would not fit next to the ring, so 32 columns per tile */
        if (epi == GD_WIDE_EPI_PLAIN && (p.N % 32u) == 0u) GD_P(2, 4, GD_WIDE_EPI_PLAIN);
        if (epi == GD_WIDE_EPI_SWIGLU && tiles != 2u && (p.swiglu_cols % 32u) == 0u && mt <= 2u) {
            if (mt == 1u) GD_P(4, 1, GD_WIDE_EPI_SWIGLU);
            GD_P(4, 2, GD_WIDE_EPI_SWIGLU);
        }
        if (epi == GD_WIDE_EPI_SWIGLU && (p.swiglu_cols % 16u) == 0u) {
            if (mt == 1u) GD_P(2, 1, GD_WIDE_EPI_SWIGLU);
            if (mt == 2u) GD_P(2, 2, GD_WIDE_EPI_SWIGLU);
            GD_P(2, 4, GD_WIDE_EPI_SWIGLU);
        }
        if (epi == GD_WIDE_EPI_ROPE && (p.rope_head_dim % 32u) == 0u && p.N == 3u * p.rope_heads * p.rope_head_dim) {
            if (mt == 1u) GD_P(2, 1, GD_WIDE_EPI_ROPE);
            if (mt == 2u) GD_P(2, 2, GD_WIDE_EPI_ROPE);
            /* 33 rows or more: the stream kernel's four workgroups per column tile are faster here (20.7 against
             * 22.3 us at 64 x 2048 -> 6144), the rotation of 64 rows weighs more than the second pass over L2 */
            return 0;
        }
    }
#undef GD_P
    if (epi == GD_WIDE_EPI_PLAIN && (p.N % 64u) == 0u) GD_W_MT(4, 4, GD_HIP_PRO_RMS_NORM, GD_WIDE_EPI_PLAIN);
    if (epi == GD_WIDE_EPI_SWIGLU && p.swiglu_cols == p.N) {
        if (tiles != 2u && (p.swiglu_cols % 32u) == 0u) GD_W_MT(4, 4, GD_HIP_PRO_RMS_NORM, GD_WIDE_EPI_SWIGLU);
        if ((p.swiglu_cols % 16u) == 0u) GD_W_MT(2, 4, GD_HIP_PRO_RMS_NORM, GD_WIDE_EPI_SWIGLU);
    }
    if (epi == GD_WIDE_EPI_ROPE && (p.rope_head_dim % 32u) == 0u && p.N == 3u * p.rope_heads * p.rope_head_dim && mt <= 2u)
        GD_W_MT(2, 4, GD_HIP_PRO_RMS_NORM, GD_WIDE_EPI_ROPE);
#endif
#undef GD_W_MT
#undef GD_W
    return 0;
}
