/*
 * F16 projections with F32 accumulation for many rows (prefill): LDS-tiled MFMA kernel for gfx950.
 *
 * Same contract and rounding points as the weight-streaming kernel in linear.hip (reference GEMMs
 * src/ops/_shared/gemm/metal_gemm_common.h:54-135 and :161-237); this one is for M >= 128 where the
 * work is bound by the matrix cores, not by weight traffic.  [N,K] weights without a prologue, whose
 * outputs take 16-byte stores, go through the kernel of linear_tile_nk.hip instead, which this file's
 * launcher asks first; here are [K,N] weights, prologues and unaligned outputs.
 *
 * Tiling.  A workgroup of 4 wavefronts (2 x 2) owns a BM x BN output tile, BM = BN = 256 or 128; a
 * wavefront owns (BM/2) x (BN/2) as WM x WN tiles of v_mfma_f32_32x32x16_f16 (4 x 4 tiles = 256
 * accumulator registers per lane for the 256 tile, one wavefront per SIMD).  Every MFMA fragment
 * (row l%32, 8 consecutive k starting at 8*(l/32)) is one 16-byte LDS read; a 4 x 4 wavefront tile reads
 * 8 fragments for 16 MFMAs.  The weight fragment is the first MFMA operand, so a lane ends up with four
 * consecutive output columns of one row per register quad (result layout of a 32x32 tile: lane l holds
 * activation row l%32; register 4q+r holds weight row 8q + 4*(l/32) + r).
 *
 * Workgroups are persistent: the grid has one workgroup per compute unit, which walks the output tiles
 * t, t + grid, ...  The operand loads of the next tile are requested before the epilogue of the current
 * one, so their latency and the epilogue's stores overlap.
 *
 * K advances in tiles of 64 through two LDS stages.  Two ways of staging:
 *  - direct (no prologue, whole tiles, K % 64 == 0): global -> LDS loads that bypass the registers, serving
 *    both weight layouts (a [K,N] weight is staged as it lies and transposed by ds_read_b64_tr_b16).  The
 *    instruction stream of a K tile is laid out by hand, see the code.
 *  - through registers (prologues, ragged tiles): the next tile's global loads are issued before the matrix
 *    instructions of the current one and stored to the other stage during its last two steps.
 * LDS has 64 banks of 4 bytes on this chip and serves 16 lanes of a 16-byte read at a time; chunk c (16
 * bytes = 8 k) of row r sits at r*8 + (c ^ swizzle(r)) with swizzles that make any 16 consecutive rows of
 * one k chunk hit all 64 banks (measured: no bank conflict cycles).
 *
 * What bounds it on MI355X: under this load the chip clocks at about 1.55 GHz (counter GRBM_GUI_ACTIVE
 * against the kernel's duration), which puts the matrix peak at about 1.6 PFLOP/s, 64 % of the published
 * 2.5 at 2.4 GHz; the vendor library reaches 1.0-1.5 PFLOP/s on the same shapes.
 *
 * Prologues are applied while the activation tile moves from registers to LDS (rounded to F16 there,
 * like the reference's separate kernels): the swiglu gate reads the second half of the row, the
 * rms_norm scale uses per-row factors computed by the workgroup before the main loop.
 *
 * Epilogue.  In WM passes of 64 rows: accumulators (+ bias, in F32 or after the F16 rounding, by mode) are
 * rounded to F16 and written as 8-byte pieces into a separate 64-row LDS buffer, then read back as 16-byte
 * row pieces and stored, adding the residual in F16.
 *
 * Tile order: workgroup ids are dealt round-robin to the 8 XCDs, so the tile index is first remapped to
 * give each XCD a contiguous run of tiles, and runs walk 8 tile rows by column so that the workgroups
 * resident on one XCD share a few activation and weight panels in its L2.
 */
#include "../../_shared/hip_device.h"
#include "hip_linear_types.h"
#include "linear_elem.h"
#include "linear_tile_nk.h"
#include <type_traits>

#define GD_TILE_BK 64u

__device__ __forceinline__ uint32_t gd_tile_slot(uint32_t row, uint32_t c)
{
    return row * 8u + (c ^ (row & 7u) ^ ((row >> 3) & 7u));
}

__device__ __forceinline__ float gd_tile_silu(float z)
{
    const float e = __expf(-fabsf(z));
    /* 1 / (1 + e) with e in (0, 1]: the reciprocal instruction is good to one unit in the last place of F32, and the
     * product is rounded to F16 afterwards; the division's dozen instructions per element would make the gated
     * epilogue of a tile a quarter longer */
    const float inv = __builtin_amdgcn_rcpf(1.0f + e);
    return z * (z >= 0.0f ? inv : e * inv);
}

__device__ __forceinline__ float gd_tile_gated(float value, float gate, const gd_hip_linear_params &p)
{
#if GD_LINEAR_IS_BF16
    if (p.flags & GD_HIP_LINEAR_CLAMPED_GATE) return gd_lin_clamped_gate(value, gate, p.gate_limit, p.gate_alpha);
    if (p.flags & GD_HIP_LINEAR_GELU_GATE) {
        const float u = 2.0f * 0.7978845608028654f * (gate + 0.044715f * gate * gate * gate);
        const float e = __expf(-fabsf(u)), inv = __builtin_amdgcn_rcpf(1.0f + e);
        return value * gate * (u >= 0.0f ? inv : e * inv);
    }
#endif
    (void)p;
    return value * gd_tile_silu(gate);
}

/* 16 bytes per lane from global memory straight into LDS: lane l's data lands at lds_base + 16*l.
 * Written as assembly because the compiler, not knowing which LDS stage a load fills, would otherwise
 * wait for ALL outstanding loads before every LDS read; the kernel counts them itself (s_waitcnt vmcnt). */
__device__ __forceinline__ void gd_tile_load_lds16(const gd_elem *uniform_base, uint32_t lane_byte_offset,
                                                   uint32_t lds_byte_address)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(lds_byte_address), "v"(lane_byte_offset), "s"(uniform_base)
                 : "memory");
}

template <int WM, int WN, bool W_NK, int PRO>
__global__ void __launch_bounds__(256)
gd_linear_tile_kernel(const gd_elem *__restrict__ x, const gd_elem *__restrict__ w, const gd_elem *__restrict__ bias,
                      const gd_elem *__restrict__ residual, const gd_elem *__restrict__ norm_w,
                      gd_elem *__restrict__ y, gd_hip_linear_params p, uint32_t tiles_m, uint32_t tiles_n,
                      uint32_t vector_store)
{
    constexpr uint32_t BM = 64u * WM, BN = 64u * WN;
    constexpr int A_PER = BM / 32;                 /* 16-byte chunks of the activation tile per thread */
    constexpr int B_PER = W_NK ? (int)(BN / 32) : 8; /* weight chunks per thread */
    constexpr uint32_t STAGE_BYTES = 2u * (BM + BN) * 8u * 16u; /* both stages of both operands */
    extern __shared__ __align__(16) unsigned char gd_tile_smem[];
    gd_elem8 *sA = reinterpret_cast<gd_elem8 *>(gd_tile_smem); /* [2][BM*8] */
    gd_elem8 *sB = sA + 2u * BM * 8u;                          /* [2][BN*8] */
    unsigned char *epi = gd_tile_smem + STAGE_BYTES;           /* [64][BN] halfs */
    float *s_inv = reinterpret_cast<float *>(epi); /* [BM] row factors of rms_norm; live during the main loop only */

    const uint32_t total = tiles_m * tiles_n;
    constexpr bool DIRECT = PRO == GD_HIP_PRO_NONE;
    uint32_t m0 = 0u, n0 = 0u; /* origin of the current tile (rows, output columns) */
    /* swiglu epilogue ([N,K] weights of 2H rows, H = p.N output columns).  The BN weight rows of a tile are two
     * wavefront columns of BN/2; each holds HW = BN/4 value rows (n0 + wc*HW ..) in its first half and the matching
     * gate rows (H + n0 + wc*HW ..) in its second half, so a lane finds value and gate of one output column in
     * its own accumulators (tiles j and j + WN/2).  The tile then owns BN/2 output columns. */
    const bool gated = p.swiglu_cols != 0u;
    const uint32_t out_bn = gated ? BN / 2u : BN;
    constexpr uint32_t HW = BN / 4u;
    auto wrow = [&](uint32_t tn0, uint32_t r) __attribute__((always_inline)) {
        const uint32_t wc = r / (BN / 2u), wr = r % (BN / 2u);
        return gated ? (wr < HW ? tn0 + wc * HW + wr : p.swiglu_cols + tn0 + wc * HW + (wr - HW)) : tn0 + r;
    };
    auto wrow_ok = [&](uint32_t tn0, uint32_t r) __attribute__((always_inline)) {
        return (gated ? tn0 + (r / (BN / 2u)) * HW + r % HW : tn0 + r) < p.N;
    };
    auto locate = [&](uint32_t t, uint32_t &tm0, uint32_t &tn0) __attribute__((always_inline)) {
        /* XCD t % 8 takes a contiguous run of tiles, one longer in the first total % 8 of them.  (Tile t as it comes, as it once was
         * where 8 does not divide the tiles, gives every XCD one row tile of each group of 8 and so 33 panels for 32 tiles instead
         * of 12: 2825 clocks per K tile against 2290 at 24576 x 4096 -> 16384, operands beyond the memory-side cache) */
        const uint32_t xcd = t & 7u, pid = xcd * (total >> 3) + min(xcd, total & 7u) + (t >> 3);
        const uint32_t width = 8u * tiles_n;
        const uint32_t first_m = (pid / width) * 8u;
        const uint32_t gsz = min(tiles_m - first_m, 8u);
        const uint32_t row_tile = first_m + (pid % width) % gsz;
        tn0 = ((pid % width) / gsz) * out_bn;
        tm0 = row_tile * BM;
    };
    auto direct_ok = [&](uint32_t tm0, uint32_t tn0) __attribute__((always_inline)) {
        return DIRECT && tm0 + BM <= p.M && tn0 + out_bn <= p.N && (p.K % 64u) == 0u && p.K >= 128u;
    };

    uint32_t tid_opaque = threadIdx.x;
    bool prefetched = false; /* the first two K tiles of the current output tile are already requested */
    for (uint32_t tile = blockIdx.x; tile < total; tile += gridDim.x) {
    /* Everything below is derived from the thread id anew for every tile: were it loop-invariant, the
     * compiler would hoist some hundred addresses and offsets out of the tile loop and spill them. */
    asm volatile("" : "+v"(tid_opaque));
    const uint32_t tid = tid_opaque, lane = tid & 63u, wave = tid >> 6;
    const uint32_t wm = wave >> 1, wn = wave & 1u;
    locate(tile, m0, n0);

    /* staging coordinates */
    const uint32_t a_c = tid & 7u, a_r = tid >> 3; /* activation: chunk a_c of rows a_r + 32*i */
    /* weight [K,N]: thread owns the 8(k) x 8(n) block (kb_j, kb_nc) of the tile */
    const uint32_t kb_per_row = BN / 8u;
    const uint32_t kb_j = tid / kb_per_row, kb_nc = tid % kb_per_row;
    constexpr bool KB_ALL = BN >= 256u; /* every thread owns a block */
    const bool kb_active = W_NK ? false : (tid < BN);

    gd_elem8 ra[A_PER], rz[PRO == GD_HIP_PRO_SWIGLU ? A_PER : 1], rb[B_PER], rn;
    const gd_elem8 zero8 = (gd_elem8)(gd_elem)0.f;
    const uint32_t ktiles = (p.K + GD_TILE_BK - 1u) / GD_TILE_BK;

    /* ---- staging through registers (any prologue, either weight layout, ragged tiles) ---------------- */
    auto load_tile = [&](uint32_t kt, auto guarded_tag) __attribute__((always_inline)) {
        constexpr bool GUARDED = decltype(guarded_tag)::value;
        const uint32_t k = kt * GD_TILE_BK + a_c * 8u;
        const bool kok = !GUARDED || k < p.K;
#pragma unroll
        for (int i = 0; i < A_PER; ++i) {
            const uint32_t gm = m0 + a_r + 32u * i;
            if (GUARDED) {
                ra[i] = zero8;
                if (PRO == GD_HIP_PRO_SWIGLU) rz[i] = zero8;
            }
            if (!GUARDED || (kok && gm < p.M)) {
                const gd_elem *xr = x + (size_t)gm * p.ldx + k;
                ra[i] = *reinterpret_cast<const gd_elem8 *>(xr);
                if (PRO == GD_HIP_PRO_SWIGLU) rz[i] = *reinterpret_cast<const gd_elem8 *>(xr + p.K);
            }
        }
        if (PRO == GD_HIP_PRO_RMS_NORM) rn = kok ? *reinterpret_cast<const gd_elem8 *>(norm_w + k) : zero8;
        if (W_NK) {
#pragma unroll
            for (int i = 0; i < B_PER; ++i) {
                const uint32_t gn = wrow(n0, a_r + 32u * (uint32_t)i);
                if (GUARDED) rb[i] = zero8;
                if (!GUARDED || (kok && wrow_ok(n0, a_r + 32u * (uint32_t)i)))
                    rb[i] = *reinterpret_cast<const gd_elem8 *>(w + (size_t)gn * p.ldw + k);
            }
        } else {
            const uint32_t gn = n0 + kb_nc * 8u;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint32_t gk = kt * GD_TILE_BK + kb_j * 8u + i;
                if (GUARDED || !KB_ALL) rb[i] = zero8;
                if ((KB_ALL || kb_active) && (!GUARDED || (gk < p.K && gn < p.N)))
                    rb[i] = *reinterpret_cast<const gd_elem8 *>(w + (size_t)gk * p.ldw + gn);
            }
        }
    };
    auto store_a = [&](uint32_t stage, int i) __attribute__((always_inline)) {
        gd_elem8 *dA = sA + stage * BM * 8u;
        const uint32_t r = a_r + 32u * i;
        gd_elem8 a = ra[i];
        if (PRO == GD_HIP_PRO_SWIGLU) {
#pragma unroll
            for (int e = 0; e < 8; ++e) a[e] = (gd_elem)((float)a[e] * gd_tile_silu((float)rz[i][e]));
        }
        if (PRO == GD_HIP_PRO_RMS_NORM) {
            const float inv = s_inv[r];
#pragma unroll
            for (int e = 0; e < 8; ++e) a[e] = (gd_elem)((float)a[e] * (float)rn[e] * inv);
        }
        dA[gd_tile_slot(r, a_c)] = a;
    };
    auto store_b = [&](uint32_t stage, int i) __attribute__((always_inline)) {
        gd_elem8 *dB = sB + stage * BN * 8u;
        if (W_NK) {
            dB[gd_tile_slot(a_r + 32u * i, a_c)] = rb[i];
        } else if (KB_ALL || kb_active) {
            gd_elem8 t; /* column i of the 8 x 8 block becomes one k-contiguous chunk */
#pragma unroll
            for (int r = 0; r < 8; ++r) t[r] = rb[r][i];
            dB[gd_tile_slot(kb_nc * 8u + i, kb_j)] = t;
        }
    };
    auto store_tile = [&](uint32_t stage) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < A_PER; ++i) store_a(stage, i);
#pragma unroll
        for (int i = 0; i < B_PER; ++i) store_b(stage, i);
    };

    /* ---- staging straight into LDS (plain activation, interior tiles) -----------------------------
     * A wavefront-wide 16-byte load writes 64 consecutive chunks = 8 rows of an LDS tile, whole 128-byte
     * lines per row; lane L fills position L%8 of row L/8 and therefore fetches the global chunk that the
     * swizzle puts there (chunk c of row r sits at r*8 + (c ^ (r & 7) ^ ((r >> 3) & 1))).  Wavefront w
     * stages rows [w*BM/4, (w+1)*BM/4) of the activation tile and the same share of the weight tile.
     *
     * A weight stored [K,N] is staged as it lies: 64 k-rows of BN halfs per stage, a wavefront load
     * filling 1024 / (2*BN) whole rows, with chunk p of k-row r at position p ^ ((r & 3) << 2).  Its
     * fragments come from ds_read_b64_tr_b16, which hands lane i of a 16-lane group element i%4 of the
     * 8-byte words addressed by lanes i/4, i/4 + 4, i/4 + 8, i/4 + 12: lane q + 4e addresses k-row e,
     * columns 4q..4q+3, so lane i receives four consecutive k of column i.  Two such reads (k 0-3, 4-7)
     * make one MFMA operand; the xor spreads the four k-rows of a read over all banks. */
    constexpr uint32_t DBK = 64u, CH = 8u, RW = 8u; /* K tile, chunks per staged row, rows per wavefront load */
    constexpr int A_DIRECT = BM / 4 / RW, B_DIRECT = BN / 4 / RW; /* loads per wavefront, K tile and operand */
    constexpr int PER_TILE = A_DIRECT + B_DIRECT;
    const uint32_t d_lane_chunk = (lane & 7u) ^ ((lane >> 3) & 7u);
    /* rows 8..15 of every 16 (odd wavefront loads) use the swizzle with bit 0 flipped */
    const uint32_t d_off_a = ((lane >> 3) * p.ldx + d_lane_chunk * 8u) * 2u; /* bytes */
    const uint32_t d_off_a1 = ((lane >> 3) * p.ldx + (d_lane_chunk ^ 1u) * 8u) * 2u;
    constexpr uint32_t CPR = BN / 8u, RPL = 64u / CPR; /* [K,N] stage: chunks per k-row, k-rows per wavefront load */
    const uint32_t d_off_b = W_NK ? ((lane >> 3) * p.ldw + d_lane_chunk * 8u) * 2u : ((lane / CPR) * p.ldw) * 2u;
    const uint32_t d_off_b1 = ((lane >> 3) * p.ldw + (d_lane_chunk ^ 1u) * 8u) * 2u;
    gd_elem8 *dA = reinterpret_cast<gd_elem8 *>(gd_tile_smem); /* [2][BM*8] */
    gd_elem8 *dB = dA + 2u * BM * CH;                          /* [2][BN*8] */
    const uint32_t wave_u = __builtin_amdgcn_readfirstlane(wave);
    const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)gd_tile_smem;
    /* item t < A_DIRECT: a wavefront load of the activation tile; A_DIRECT <= t: one of the weight tile */
    auto direct_load_item = [&](uint32_t tm0, uint32_t tn0, uint32_t kt, uint32_t t) __attribute__((always_inline)) {
        const uint32_t stage = kt & 1u;
        if (t < (uint32_t)A_DIRECT) {
            const uint32_t row0 = wave_u * (BM / 4u) + t * RW;
            gd_tile_load_lds16(x + (size_t)(tm0 + row0) * p.ldx + kt * DBK, (t & 1u) ? d_off_a1 : d_off_a,
                               lds_base + (stage * BM * CH + row0 * CH) * 16u);
        } else if (W_NK) {
            const uint32_t tb = t - (uint32_t)A_DIRECT;
            const uint32_t row0 = wave_u * (BN / 4u) + tb * RW;
            gd_tile_load_lds16(w + (size_t)wrow(tn0, row0) * p.ldw + kt * DBK, (tb & 1u) ? d_off_b1 : d_off_b,
                               lds_base + ((2u * BM + stage * BN) * CH + row0 * CH) * 16u);
        } else {
            /* k-rows kr0 .. kr0+RPL-1 of the tile; lane L fills position L%CPR of row kr0 + L/CPR */
            const uint32_t tb = t - (uint32_t)A_DIRECT;
            const uint32_t kr0 = (wave_u * (uint32_t)B_DIRECT + tb) * RPL;
            const uint32_t row = (RPL >= 4u ? 0u : ((tb * RPL) & 3u)) + lane / CPR; /* row & 3 */
            const uint32_t chunk = (lane % CPR) ^ ((row & 3u) << 2);
            gd_tile_load_lds16(w + (size_t)(kt * DBK + kr0) * p.ldw + tn0, d_off_b + chunk * 16u,
                               lds_base + ((2u * BM + stage * BN) * CH + kr0 * CPR) * 16u);
        }
    };
    auto direct_loads = [&](uint32_t tm0, uint32_t tn0, uint32_t kt) __attribute__((always_inline)) {
#pragma unroll
        for (uint32_t t = 0; t < (uint32_t)PER_TILE; ++t) direct_load_item(tm0, tn0, kt, t);
    };

    gd_float16 acc[WM][WN];

    const uint32_t frag_row = lane & 31u, frag_c = lane >> 5;
    const uint32_t a_frag_row = wm * (WM * 32u) + frag_row, b_frag_row = wn * (WN * 32u) + frag_row;

    auto load_frags = [&](const gd_elem8 *cA, const gd_elem8 *cB, uint32_t ks, gd_elem8 (&fa)[WM], gd_elem8 (&fb)[WN])
        __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < WM; ++i) fa[i] = cA[gd_tile_slot(a_frag_row + i * 32u, ks * 2u + frag_c)];
#pragma unroll
        for (int j = 0; j < WN; ++j) fb[j] = cB[gd_tile_slot(b_frag_row + j * 32u, ks * 2u + frag_c)];
    };
    auto multiply = [&](const gd_elem8 (&fa)[WM], const gd_elem8 (&fb)[WN]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < WM; ++i)
#pragma unroll
            for (int j = 0; j < WN; ++j)
                acc[i][j] = GD_MFMA_32X32X16(fb[j], fa[i], acc[i][j]);
    };

    constexpr uint32_t STEPS = GD_TILE_BK / 16u;
    /* Register path, one K tile of 4 steps of 16: the fragments of step s+1 are read while the matrix cores
     * work on step s; the next tile's global loads are issued first and stored to the other LDS stage
     * during the last two steps. */
    auto k_tile_regs = [&](uint32_t kt, auto guarded_tag, auto more_tag) __attribute__((always_inline)) {
        constexpr bool MORE = decltype(more_tag)::value;
        const uint32_t stage = kt & 1u;
        const gd_elem8 *cA = sA + stage * BM * 8u, *cB = sB + stage * BN * 8u;
        gd_elem8 fa[2][WM], fb[2][WN];
        load_frags(cA, cB, 0u, fa[0], fb[0]);
        if (MORE) load_tile(kt + 1u, guarded_tag);
#pragma unroll
        for (uint32_t ks = 0; ks < STEPS; ++ks) {
            if (ks + 1u < STEPS) load_frags(cA, cB, ks + 1u, fa[(ks + 1u) & 1u], fb[(ks + 1u) & 1u]);
            multiply(fa[ks & 1u], fb[ks & 1u]);
            if (MORE && ks >= STEPS - 2u) {
                const int half = (int)(ks - (STEPS - 2u));
#pragma unroll
                for (int i = half * (A_PER / 2); i < (half + 1) * (A_PER / 2); ++i) store_a(stage ^ 1u, i);
#pragma unroll
                for (int i = half * (B_PER / 2); i < (half + 1) * (B_PER / 2); ++i) store_b(stage ^ 1u, i);
            }
        }
        __syncthreads();
    };

    auto direct_frag_a = [&](const gd_elem8 *cA, uint32_t ks, uint32_t i) __attribute__((always_inline)) {
        const uint32_t c = ks * 2u + frag_c;
        const uint32_t r = a_frag_row + i * 32u;
        return cA[r * CH + (c ^ (r & 7u) ^ ((r >> 3) & 1u))];
    };
    auto direct_frag_b = [&](const gd_elem8 *cB, uint32_t ks, uint32_t j) __attribute__((always_inline)) {
        if (W_NK) {
            const uint32_t c = ks * 2u + frag_c;
            const uint32_t r = b_frag_row + j * 32u;
            return cB[r * CH + (c ^ (r & 7u) ^ ((r >> 3) & 1u))];
        } else {
            /* lane l = 16g + (q + 4e): k-rows ks*16 + 8*(g/2) + e (+4 for the second read), columns
             * 16*(g%2) + 4q .. +3 of this 32-column block */
            const uint32_t g = lane >> 4, q = lane & 3u, e = (lane >> 2) & 3u;
            const uint32_t col = wn * (WN * 32u) + j * 32u + 16u * (g & 1u) + 4u * q;
            const uint32_t krow = ks * 16u + 8u * (g >> 1) + e; /* krow & 3 == e for both reads */
            const uint32_t byte0 = krow * (BN * 2u) + (((col >> 3) ^ (e << 2)) << 4) + (q & 1u) * 8u;
            const unsigned char *base = reinterpret_cast<const unsigned char *>(cB);
            typedef short gd_short4 __attribute__((ext_vector_type(4)));
            const gd_short4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (__attribute__((address_space(3))) gd_short4 *)(base + byte0));
            const gd_short4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (__attribute__((address_space(3))) gd_short4 *)(base + byte0 + 4u * (BN * 2u)));
            union { gd_short4 s[2]; gd_elem8 h; } u;
            u.s[0] = lo;
            u.s[1] = hi;
            return u.h;
        }
    };
    /* Direct path, one wavefront's instruction stream for a K tile (4 steps of 16 matrix instructions),
     * pinned with scheduling barriers: every matrix instruction is followed by at most one fragment read or
     * one global -> LDS load, so the matrix pipe never waits for an LDS round trip.
     *   steps 0-2 of tile kt: their first matrix instructions are followed by the fragment reads of the next
     *   step (into the other register set);
     *   step 3: wait for this wavefront's loads of tile kt+1, barrier (tile kt+1 visible to all, stage kt%2
     *           read by all), then read step 0 of tile kt+1 and, behind the later matrix instructions,
     *           request the first half of tile kt+2 into the freed stage; step 0 of the next tile requests
     *           the second half.
     * TAIL 0: steady state; 1: tile kt+1 exists but not kt+2; 2: last tile. */
    gd_elem8 qa[2][WM], qb[2][WN];
    constexpr uint32_t NM = WM * WN, NR = WM + WN, NL = PER_TILE / 2;
    constexpr uint32_t RPM = NM >= 2u * NR ? 1u : (2u * NR + NM - 1u) / NM; /* fragment reads per matrix instruction */
    constexpr uint32_t LPM = NM >= 2u * NL ? 1u : (2u * NL + NM - 1u) / NM; /* loads per matrix instruction */
    auto direct_step = [&](uint32_t kt, auto ks_tag, auto tail_tag) __attribute__((always_inline)) {
        constexpr uint32_t KS = decltype(ks_tag)::value;
        constexpr int TAIL = decltype(tail_tag)::value;
        constexpr uint32_t CUR = KS & 1u, NXT = CUR ^ 1u;
        constexpr bool READS = KS < 3u || TAIL < 2;
        constexpr bool LOADS = (KS == 3u && TAIL == 0) || (KS == 0u && TAIL < 2);
        const uint32_t rstage = KS < 3u ? (kt & 1u) : ((kt + 1u) & 1u);
        const gd_elem8 *cA = dA + rstage * BM * CH, *cB = dB + rstage * BN * CH;
        const uint32_t rks = KS < 3u ? KS + 1u : 0u;
        const bool loads_on = KS == 3u || kt >= 1u; /* tiles 0 and 1 are requested before the loop */
        if (KS == 3u && TAIL < 2) {
            __builtin_amdgcn_s_waitcnt(0x0070); /* vmcnt(0) lgkmcnt(0) */
            __syncthreads();
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (uint32_t idx = 0; idx < NM; ++idx) {
            const uint32_t i = idx / WN, j = idx % WN;
            acc[i][j] = GD_MFMA_32X32X16(qb[CUR][j], qa[CUR][i], acc[i][j]);
            if (READS) {
#pragma unroll
                for (uint32_t r = min(idx * RPM, NR); r < min((idx + 1u) * RPM, NR); ++r) {
                    /* a0 b0 a1 b1 ...: the order in which the next step consumes them; behind the shorter of the
                     * two lists the rest of the longer one */
                    constexpr uint32_t BOTH = 2u * (WM < WN ? WM : WN);
                    if (r >= BOTH) {
                        if constexpr (WM > WN) qa[NXT][r - BOTH / 2u] = direct_frag_a(cA, rks, r - BOTH / 2u);
                        else qb[NXT][r - BOTH / 2u] = direct_frag_b(cB, rks, r - BOTH / 2u);
                    } else if ((r & 1u) == 0u) qa[NXT][r >> 1] = direct_frag_a(cA, rks, r >> 1);
                    else qb[NXT][r >> 1] = direct_frag_b(cB, rks, r >> 1);
                }
            }
            constexpr uint32_t LI = (NL + LPM - 1u) / LPM; /* matrix instructions that carry loads */
            if (LOADS && loads_on && idx >= NM - LI) {
#pragma unroll
                for (uint32_t t = (idx - (NM - LI)) * LPM; t < min((idx - (NM - LI) + 1u) * LPM, NL); ++t)
                    direct_load_item(m0, n0, KS == 3u ? kt + 2u : kt + 1u, KS == 3u ? t : NL + t);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto k_tile_direct = [&](uint32_t kt, auto tail_tag) __attribute__((always_inline)) {
        direct_step(kt, std::integral_constant<uint32_t, 0>{}, tail_tag);
        direct_step(kt, std::integral_constant<uint32_t, 1>{}, tail_tag);
        direct_step(kt, std::integral_constant<uint32_t, 2>{}, tail_tag);
        direct_step(kt, std::integral_constant<uint32_t, 3>{}, tail_tag);
    };
    using gd_t = std::true_type;
    using gd_f = std::false_type;

    /* 8-byte pieces of the epilogue buffer: piece u of row e sits at e*EU + (u ^ (e & 31)), which spreads the
     * 32 rows that one wavefront store touches over all banks; a 16-byte read-back takes pieces 2v, 2v+1 */
    constexpr uint32_t EU = BN / 4u;
    gd_elem4 bq[WN][4]; /* bias of the 4 columns of every register quad, loaded once per tile */
    auto load_bias = [&]() __attribute__((always_inline)) {
        const bool vec = (reinterpret_cast<uintptr_t>(bias) & 7u) == 0u;
#pragma unroll
        for (int j = 0; j < WN; ++j) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t lc = wn * (WN * 32u) + (uint32_t)j * 32u + 8u * (uint32_t)q + 4u * frag_c;
                const uint32_t gc = wrow(n0, lc); /* the four columns of a quad lie in the same half of a gated tile */
                if (vec && (gc & 3u) == 0u && wrow_ok(n0, lc + 3u)) {
                    bq[j][q] = *reinterpret_cast<const gd_elem4 *>(bias + gc);
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        bq[j][q][r] = wrow_ok(n0, lc + (uint32_t)r) ? bias[gc + (uint32_t)r] : (gd_elem)0.f;
                }
            }
        }
    };
    /* the four columns of register quad q of accumulator tile a, rounded to F16 with the bias of the mode */
    auto quad_f16 = [&](auto mode_tag, const gd_float16 &a, int j, int q) __attribute__((always_inline)) {
        constexpr uint32_t MODE = decltype(mode_tag)::value;
        gd_elem4 h;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float v = a[4 * q + r];
#if GD_LINEAR_IS_BF16
            if (p.flags & GD_HIP_LINEAR_SQUARE_RELU) {
                h[r] = (gd_elem)gd_lin_activated(MODE == GD_HIP_EPI_BIAS_F32 ? v + (float)bq[j][q][r] : v, p.flags);
                continue;
            }
#endif
            if (MODE == GD_HIP_EPI_NONE) h[r] = (gd_elem)v;
            else if (MODE == GD_HIP_EPI_BIAS_F32) h[r] = (gd_elem)(v + (float)bq[j][q][r]);
            else h[r] = (gd_elem)v + bq[j][q][r];
        }
        return h;
    };
#if GD_LINEAR_IS_BF16
    auto quad_gated = [&](auto mode_tag, const gd_float16 &value, const gd_float16 &gate, int j, int q) __attribute__((always_inline)) {
        gd_elem4 h;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            float fv = value[4 * q + t], fg = gate[4 * q + t];
            if (decltype(mode_tag)::value == GD_HIP_EPI_BIAS_F32) {
                fv += (float)bq[j][q][t];
                fg += (float)bq[j + WN / 2][q][t];
            }
            h[t] = (gd_elem)gd_tile_gated(fv, fg, p);
        }
        return h;
    };
#endif
    auto epilogue_pass = [&](auto pass_tag, auto mode_tag) __attribute__((always_inline)) {
        constexpr int I = decltype(pass_tag)::value;
        const uint32_t e = wm * 32u + frag_row;
#if GD_LINEAR_IS_BF16
        /* gated from the F32 sums, as in a whole tile: which tile a row lies in does not show in its bits */
        constexpr int STAGED = WN / 2;
#else
        constexpr int STAGED = WN;
#endif
#pragma unroll
        for (int j = 0; j < WN; ++j) {
            if (gated && j >= STAGED) break;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t lc = wn * (WN * 32u) + (uint32_t)j * 32u + 8u * (uint32_t)q + 4u * frag_c;
                gd_elem4 h;
#if GD_LINEAR_IS_BF16
                if (gated && j < WN / 2) h = quad_gated(mode_tag, acc[I][j], acc[I][(j + WN / 2) % WN], j, q);
                else
#endif
                h = quad_f16(mode_tag, acc[I][j], j, q);
                *reinterpret_cast<gd_elem4 *>(epi + (e * EU + ((lc >> 2) ^ (e & 31u))) * 8u) = h;
            }
        }
        __syncthreads();
        constexpr uint32_t CPRW = BN / 8u; /* 16-byte chunks per row */
        auto read_chunk = [&](uint32_t er, uint32_t v) __attribute__((always_inline)) {
            const uint32_t xr = er & 31u;
            const gd_elem8 raw = *reinterpret_cast<const gd_elem8 *>(epi + (er * EU + 2u * (v ^ (xr >> 1))) * 8u);
            gd_elem8 h = raw;
            if (xr & 1u) {
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    h[t] = raw[4 + t];
                    h[4 + t] = raw[t];
                }
            }
            return h;
        };
        if (gated) {
            /* a value chunk and the gate chunk HW/8 behind it make one output chunk (F16; BF16: multiplied already) */
#pragma unroll
            for (uint32_t idx0 = 0; idx0 < 32u * CPRW; idx0 += 256u) {
                const uint32_t idx = idx0 + tid;
                const uint32_t er = idx / (CPRW / 2u), v = idx % (CPRW / 2u);
                const uint32_t gr = m0 + (er >> 5) * (WM * 32u) + (uint32_t)I * 32u + (er & 31u), gc = n0 + v * 8u;
                if (gr >= p.M || gc >= p.N) continue;
                /* staged columns: wavefront column wc holds its HW value columns, then their gates */
                const uint32_t cv = (v / (HW / 8u)) * (HW / 4u) + v % (HW / 8u);
                gd_elem8 h = read_chunk(er, cv);
#if !GD_LINEAR_IS_BF16
                const gd_elem8 hg = read_chunk(er, cv + HW / 8u);
#pragma unroll
                for (int t = 0; t < 8; ++t) h[t] = (gd_elem)gd_tile_gated((float)h[t], (float)hg[t], p);
#endif
                gd_elem *yr = y + (size_t)gr * p.ldy + gc;
                if (vector_store && gc + 8u <= p.N) {
                    *reinterpret_cast<gd_elem8 *>(yr) = h;
                } else {
                    for (uint32_t t = 0; t < 8u && gc + t < p.N; ++t) yr[t] = h[t];
                }
            }
        } else {
#pragma unroll
        for (uint32_t idx0 = 0; idx0 < 64u * CPRW; idx0 += 256u) {
            const uint32_t idx = idx0 + tid;
            const uint32_t er = idx / CPRW, v = idx % CPRW;
            const uint32_t gr = m0 + (er >> 5) * (WM * 32u) + (uint32_t)I * 32u + (er & 31u), gc = n0 + v * 8u;
            if (gr >= p.M || gc >= p.N) continue;
            gd_elem8 h = read_chunk(er, v);
            gd_elem *yr = y + (size_t)gr * p.ldy + gc;
            if (vector_store && gc + 8u <= p.N) {
                if (p.has_residual) {
                    const gd_elem8 r = *reinterpret_cast<const gd_elem8 *>(residual + (size_t)gr * p.ldr + gc);
#pragma unroll
                    for (int t = 0; t < 8; ++t) h[t] = r[t] + h[t];
                }
                /* long K: the output is not read again soon and would only push operand panels out of L2 */
                if (p.K >= 1024u) __builtin_nontemporal_store(h, reinterpret_cast<gd_elem8 *>(yr));
                else *reinterpret_cast<gd_elem8 *>(yr) = h;
            } else {
                for (uint32_t t = 0; t < 8u && gc + t < p.N; ++t) {
                    gd_elem v1 = h[t];
                    if (p.has_residual) v1 = residual[(size_t)gr * p.ldr + gc + t] + v1;
                    yr[t] = v1;
                }
            }
        }
        }
        if (I + 1 < WM) __syncthreads(); /* the next pass overwrites the buffer; after the last pass the barriers
                                            of the next tile's main loop come first */
    };
    auto epilogue = [&](auto mode_tag) __attribute__((always_inline)) {
        if (decltype(mode_tag)::value != GD_HIP_EPI_NONE) load_bias();
        epilogue_pass(std::integral_constant<int, 0>{}, mode_tag);
        epilogue_pass(std::integral_constant<int, 1>{}, mode_tag);
        if (WM > 2) epilogue_pass(std::integral_constant<int, (WM > 2 ? 2 : 0)>{}, mode_tag);
        if (WM > 3) epilogue_pass(std::integral_constant<int, (WM > 3 ? 3 : 0)>{}, mode_tag);
    };

    /* Epilogue of a whole 256-column tile whose rows can take 16-byte stores: no workgroup barriers.  A wavefront
     * rounds its own 32 x 128 block of a pass, brings the two 8-byte pieces that lanes l and l + 32 hold of one
     * 16-byte chunk into one lane (v_permlane32_swap), writes whole chunks into its own quarter of the buffer and
     * reads them back as row pieces (16 lanes x 16 bytes per row, four rows per instruction; gated tiles, whose
     * wavefront has already multiplied value and gate in registers: 8 lanes per row, eight rows).  LDS operations
     * of one wavefront are carried out in order, so the next pass overwrites the quarter without a barrier.
     * Chunk c of row e sits at e*16 + (c ^ (e & 15)) (gated: e*8 + (c ^ ((e >> 1) & 7))): 16 consecutive rows of
     * one chunk, and the lanes of one read, hit all banks.  The residual rows of a pass are requested before its
     * accumulators are rounded, so that their latency passes behind that work. */
    typedef unsigned gd_uint2v __attribute__((ext_vector_type(2)));
    auto pair_chunk = [&](gd_elem4 a, gd_elem4 b) __attribute__((always_inline)) {
        union { gd_elem4 h; uint32_t u[2]; } ua, ub;
        ua.h = a;
        ub.h = b;
        /* lanes 32-63 of the first operand change places with lanes 0-31 of the second */
        const gd_uint2v s0 = __builtin_amdgcn_permlane32_swap(ua.u[0], ub.u[0], false, false);
        const gd_uint2v s1 = __builtin_amdgcn_permlane32_swap(ua.u[1], ub.u[1], false, false);
        union { uint32_t u[4]; gd_elem8 h; } c;
        c.u[0] = s0[0];
        c.u[1] = s1[0];
        c.u[2] = s0[1];
        c.u[3] = s1[1];
        return c.h;
    };
    /* Streaming stores where the launcher asks for them: all compute units end their tiles together, and 128 KB from each of them
     * would wait for the write-back of as many dirty lines of the L2s (a launch without any store is a tenth shorter).  BF16, us:
     * 30229 x 2048 -> 11264 1174 -> 1133, 27000 x 4096 -> 16896 3106 -> 2967 */
    auto store_rows = [&](const auto &h, gd_elem *at, uint32_t step) __attribute__((always_inline)) {
        constexpr uint32_t ROWS = sizeof(h) / sizeof(h[0]);
        if (p.flags & GD_HIP_LINEAR_STREAM_Y) {
            asm volatile("; streaming"); /* the compiler makes one ordinary store of two that differ in the hint alone */
#pragma unroll
            for (uint32_t r = 0; r < ROWS; ++r) __builtin_nontemporal_store(h[r], reinterpret_cast<gd_elem8 *>(at + r * step));
            asm volatile("; streamed");
        } else {
#pragma unroll
            for (uint32_t r = 0; r < ROWS; ++r) *reinterpret_cast<gd_elem8 *>(at + r * step) = h[r];
        }
    };
    auto epilogue_own = [&](auto mode_tag) __attribute__((always_inline)) {
        if (decltype(mode_tag)::value != GD_HIP_EPI_NONE) load_bias();
        unsigned char *own = epi + wave * 8192u;
        const uint32_t rr = lane >> 4, v = lane & 15u;
        /* offsets of this lane's piece from the tile's first element; the pass and the row group add a uniform
         * term */
        const gd_elem *rtile = residual + ((size_t)m0 * p.ldr + n0);
        gd_elem *ytile = y + ((size_t)m0 * p.ldy + n0);
        const uint32_t y_lane = (wm * (WM * 32u) + rr) * p.ldy + wn * (WN * 32u) + v * 8u;
        const uint32_t r_lane = (wm * (WM * 32u) + rr) * p.ldr + wn * (WN * 32u) + v * 8u;
        auto pass = [&](auto pass_tag) __attribute__((always_inline)) {
            constexpr int I = decltype(pass_tag)::value;
            gd_elem8 res[8];
            if (p.has_residual) {
#pragma unroll
                for (uint32_t it = 0; it < 8u; ++it)
                    res[it] = *reinterpret_cast<const gd_elem8 *>(rtile + ((uint32_t)I * 32u + it * 4u) * p.ldr + r_lane);
            }
#pragma unroll
            for (int j = 0; j < WN; ++j) {
#pragma unroll
                for (int pr = 0; pr < 2; ++pr) {
                    const uint32_t c = (uint32_t)j * 4u + 2u * (uint32_t)pr + frag_c;
                    *reinterpret_cast<gd_elem8 *>(own + (frag_row * 16u + (c ^ (frag_row & 15u))) * 16u) =
                        pair_chunk(quad_f16(mode_tag, acc[I][j], j, 2 * pr), quad_f16(mode_tag, acc[I][j], j, 2 * pr + 1));
                }
            }
            gd_elem8 h[8];
#pragma unroll
            for (uint32_t it = 0; it < 8u; ++it) {
                const uint32_t e = it * 4u + rr;
                h[it] = *reinterpret_cast<const gd_elem8 *>(own + (e * 16u + (v ^ (e & 15u))) * 16u);
            }
#pragma unroll
            for (uint32_t it = 0; it < 8u; ++it) {
                if (p.has_residual) {
#pragma unroll
                    for (int t = 0; t < 8; ++t) h[it][t] = res[it][t] + h[it][t];
                }
            }
            store_rows(h, ytile + (uint32_t)I * 32u * p.ldy + y_lane, 4u * p.ldy);
        };
        pass(std::integral_constant<int, 0>{});
        pass(std::integral_constant<int, 1>{});
        if (WM > 2) pass(std::integral_constant<int, (WM > 2 ? 2 : 0)>{});
        if (WM > 3) pass(std::integral_constant<int, (WM > 3 ? 3 : 0)>{});
    };
    auto epilogue_own_gated = [&](auto mode_tag) __attribute__((always_inline)) {
        if (decltype(mode_tag)::value != GD_HIP_EPI_NONE) load_bias();
        unsigned char *own = epi + wave * 8192u;
        const uint32_t rr = lane >> 3, v = lane & 7u;
        gd_elem *ytile = y + ((size_t)m0 * p.ldy + n0);
        const uint32_t y_lane = (wm * (WM * 32u) + rr) * p.ldy + wn * HW + v * 8u;
        auto pass = [&](auto pass_tag) __attribute__((always_inline)) {
            constexpr int I = decltype(pass_tag)::value;
#pragma unroll
            for (int j = 0; j < WN / 2; ++j) {
#pragma unroll
                for (int pr = 0; pr < 2; ++pr) {
                    gd_elem4 o[2];
#pragma unroll
                    for (int s2 = 0; s2 < 2; ++s2) {
#if GD_LINEAR_IS_BF16
                        o[s2] = quad_gated(mode_tag, acc[I][j], acc[I][j + WN / 2], j, 2 * pr + s2);
#else
                        const gd_elem4 hv = quad_f16(mode_tag, acc[I][j], j, 2 * pr + s2);
                        const gd_elem4 hg = quad_f16(mode_tag, acc[I][j + WN / 2], j + WN / 2, 2 * pr + s2);
#pragma unroll
                        for (int t = 0; t < 4; ++t) o[s2][t] = (gd_elem)((float)hv[t] * gd_tile_silu((float)hg[t]));
#endif
                    }
                    const uint32_t c = (uint32_t)j * 4u + 2u * (uint32_t)pr + frag_c;
                    *reinterpret_cast<gd_elem8 *>(own + (frag_row * 8u + (c ^ ((frag_row >> 1) & 7u))) * 16u) =
                        pair_chunk(o[0], o[1]);
                }
            }
            gd_elem8 h[4];
#pragma unroll
            for (uint32_t it = 0; it < 4u; ++it) {
                const uint32_t e = it * 8u + rr;
                h[it] = *reinterpret_cast<const gd_elem8 *>(own + (e * 8u + (v ^ ((e >> 1) & 7u))) * 16u);
            }
            store_rows(h, ytile + (uint32_t)I * 32u * p.ldy + y_lane, 8u * p.ldy);
        };
        pass(std::integral_constant<int, 0>{});
        pass(std::integral_constant<int, 1>{});
        if (WM > 2) pass(std::integral_constant<int, (WM > 2 ? 2 : 0)>{});
        if (WM > 3) pass(std::integral_constant<int, (WM > 3 ? 3 : 0)>{});
    };

        /* interior tile: every staged chunk is in range, so the main loop carries no guards */
        const bool interior = m0 + BM <= p.M && n0 + out_bn <= p.N && (p.K % GD_TILE_BK) == 0u;

        if (PRO == GD_HIP_PRO_RMS_NORM) {
            __syncthreads(); /* the previous tile's epilogue has left the buffer that holds the row factors */
            for (uint32_t r = wave; r < BM; r += 4u) {
                const uint32_t row = min(m0 + r, p.M - 1u);
                const gd_elem *xr = x + (size_t)row * p.ldx;
                float ss = 0.f;
                for (uint32_t k = lane * 8u; k < p.K; k += 512u) {
                    const gd_elem8 v = *reinterpret_cast<const gd_elem8 *>(xr + k);
#pragma unroll
                    for (int e = 0; e < 8; ++e) ss = fmaf((float)v[e], (float)v[e], ss);
                }
                ss = gd_wave_sum(ss);
                if (lane == 0u) s_inv[r] = rsqrtf(ss / (float)p.K + p.eps);
            }
            __syncthreads();
        }

#pragma unroll
        for (int i = 0; i < WM; ++i)
#pragma unroll
            for (int j = 0; j < WN; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

        if (direct_ok(m0, n0)) {
            const uint32_t dtiles = p.K / 64u; /* >= 2 */
            if (!prefetched) {
                direct_loads(m0, n0, 0u);
                direct_loads(m0, n0, 1u);
            }
            /* at most PER_TILE vector memory operations outstanding: loads complete in order, so K tile 0 has
             * landed whatever else (K tile 1, stores of the previous epilogue) is still on its way */
            __builtin_amdgcn_s_waitcnt(0x0F70 | (PER_TILE & 15) | ((PER_TILE >> 4) << 14));
            __syncthreads();
            {
#pragma unroll
                for (int i = 0; i < WM; ++i) qa[0][i] = direct_frag_a(dA, 0u, (uint32_t)i);
#pragma unroll
                for (int j = 0; j < WN; ++j) qb[0][j] = direct_frag_b(dB, 0u, (uint32_t)j);
            }
            uint32_t kt = 0;
            for (; kt + 2u < dtiles; ++kt) k_tile_direct(kt, std::integral_constant<int, 0>{});
            k_tile_direct(kt, std::integral_constant<int, 1>{});
            k_tile_direct(kt + 1u, std::integral_constant<int, 2>{});
            __syncthreads(); /* every wavefront has read its last fragments: both stages are free */
            /* request the next output tile's first two K tiles now; they land during the epilogue */
            prefetched = false;
            const uint32_t next = tile + gridDim.x;
            if (next < total) {
                uint32_t nm0, nn0;
                locate(next, nm0, nn0);
                if (direct_ok(nm0, nn0)) {
                    direct_loads(nm0, nn0, 0u);
                    direct_loads(nm0, nn0, 1u);
                    prefetched = true;
                }
            }
        } else {
            prefetched = false;
            load_tile(0u, gd_t{});
            store_tile(0u);
            __syncthreads();
            if (interior) {
                for (uint32_t kt = 0; kt + 1u < ktiles; ++kt) k_tile_regs(kt, gd_f{}, gd_t{});
                k_tile_regs(ktiles - 1u, gd_f{}, gd_f{});
            } else {
                for (uint32_t kt = 0; kt + 1u < ktiles; ++kt) k_tile_regs(kt, gd_t{}, gd_t{});
                k_tile_regs(ktiles - 1u, gd_t{}, gd_f{});
            }
        }

        auto finish = [&](auto mode_tag) __attribute__((always_inline)) {
            if (WM == 4 && WN == 4 && vector_store && m0 + BM <= p.M && n0 + out_bn <= p.N) {
                if (gated) epilogue_own_gated(mode_tag);
                else epilogue_own(mode_tag);
            } else {
                epilogue(mode_tag);
            }
        };
        if (p.epilogue == GD_HIP_EPI_BIAS_F32) finish(std::integral_constant<uint32_t, GD_HIP_EPI_BIAS_F32>{});
        else if (p.epilogue == GD_HIP_EPI_BIAS_F16) finish(std::integral_constant<uint32_t, GD_HIP_EPI_BIAS_F16>{});
        else finish(std::integral_constant<uint32_t, GD_HIP_EPI_NONE>{});
    }
}

template <int WM, int WN, bool W_NK, int PRO>
int gd_linear_tile_launch_one(hipStream_t stream, const gd_elem *x, const gd_elem *w, const gd_elem *bias,
                           const gd_elem *residual, const gd_elem *norm_w, gd_elem *y, const gd_hip_linear_params &p,
                           uint32_t vector_store, uint32_t workgroups)
{
    constexpr uint32_t BM = 64u * WM, BN = 64u * WN;
    constexpr size_t lds = (size_t)2u * (BM + BN) * 8u * 16u + (size_t)64u * BN * 2u; /* stages + epilogue rows */
    static bool configured = false;
    auto kernel = gd_linear_tile_kernel<WM, WN, W_NK, PRO>;
    if (!configured) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return (int)e;
        configured = true;
    }
    const uint32_t out_bn = p.swiglu_cols != 0u ? BN / 2u : BN; /* output columns per tile */
    const uint32_t tiles_m = (p.M + BM - 1u) / BM, tiles_n = (p.N + out_bn - 1u) / out_bn;
    /* persistent workgroups: at most `workgroups` of them (a multiple of 8 keeps the tile -> XCD relation) */
    const uint32_t grid = tiles_m * tiles_n < workgroups ? tiles_m * tiles_n : workgroups;
    kernel<<<grid, 256, lds, stream>>>(x, w, bias, residual, norm_w, y, p, tiles_m, tiles_n, vector_store);
    return (int)hipGetLastError();
}

/* The F16 instantiations take minutes to compile; they are spread over translation units of their own
 * (linear_tile_part*.hip define GD_LINEAR_TILE_PART and include this file) and only declared here. */
#define GD_TILE_FORM(WORD, WM, WN, NK, PRO)                                                                              \
    WORD template int gd_linear_tile_launch_one<WM, WN, NK, PRO>(hipStream_t, const gd_elem *, const gd_elem *,          \
                                                                 const gd_elem *, const gd_elem *, const gd_elem *,      \
                                                                 gd_elem *, const gd_hip_linear_params &, uint32_t, uint32_t);
#define GD_TILE_PROLOGUES(WORD, WM, WN, NK)            \
    GD_TILE_FORM(WORD, WM, WN, NK, GD_HIP_PRO_NONE)    \
    GD_TILE_FORM(WORD, WM, WN, NK, GD_HIP_PRO_SWIGLU)  \
    GD_TILE_FORM(WORD, WM, WN, NK, GD_HIP_PRO_RMS_NORM)
#if defined(GD_LINEAR_TILE_PART) && GD_LINEAR_TILE_PART == 1
GD_TILE_PROLOGUES(, 4, 4, true)
#elif defined(GD_LINEAR_TILE_PART) && GD_LINEAR_TILE_PART == 2
GD_TILE_PROLOGUES(, 4, 4, false)
#elif defined(GD_LINEAR_TILE_PART) && GD_LINEAR_TILE_PART == 3
GD_TILE_PROLOGUES(, 2, 2, true)
GD_TILE_PROLOGUES(, 2, 2, false)
#else
#if !GD_LINEAR_IS_BF16
GD_TILE_PROLOGUES(extern, 4, 4, true)
GD_TILE_PROLOGUES(extern, 4, 4, false)
GD_TILE_PROLOGUES(extern, 2, 2, true)
GD_TILE_PROLOGUES(extern, 2, 2, false)
#endif

template <int WM, int WN>
static int launch_tile(hipStream_t stream, const gd_elem *x, const gd_elem *w, const gd_elem *bias,
                       const gd_elem *residual, const gd_elem *norm_w, gd_elem *y, const gd_hip_linear_params &p,
                       uint32_t vector_store, uint32_t workgroups)
{
#define GD_GO(NK, PRO) return gd_linear_tile_launch_one<WM, WN, NK, PRO>(stream, x, w, bias, residual, norm_w, y, p, vector_store, workgroups)
#if GD_LINEAR_IS_BF16
    GD_GO(true, GD_HIP_PRO_NONE);
#else
    if (p.w_is_nk) {
        if (p.prologue == GD_HIP_PRO_SWIGLU) GD_GO(true, GD_HIP_PRO_SWIGLU);
        if (p.prologue == GD_HIP_PRO_RMS_NORM) GD_GO(true, GD_HIP_PRO_RMS_NORM);
        GD_GO(true, GD_HIP_PRO_NONE);
    }
    if (p.prologue == GD_HIP_PRO_SWIGLU) GD_GO(false, GD_HIP_PRO_SWIGLU);
    if (p.prologue == GD_HIP_PRO_RMS_NORM) GD_GO(false, GD_HIP_PRO_RMS_NORM);
    GD_GO(false, GD_HIP_PRO_NONE);
#endif
#undef GD_GO
}

/* linear_tile_nk.hip: [N,K] weights without a prologue */
extern "C" int GD_LINEAR_FN(gd_hip_try_launch_linear_tile_nk)(hipStream_t stream, const void *x, const void *w, const void *bias,
                                                const void *residual, void *y, const gd_hip_linear_params *params,
                                                int vector_store, uint32_t units);

/* Requires: K % 8 == 0, 16-byte aligned x rows (and gate half), w rows (for [K,N]: N % 8 == 0 too) and
 * norm weight; M >= 1.  big_tiles: use the 256 x 256 tile (one workgroup per compute unit; the 128 x 128 tile
 * fits two). */
extern "C" int GD_LINEAR_FN(gd_hip_launch_linear_tile)(hipStream_t stream, const void *x, const void *w, const void *bias,
                                         const void *residual, const void *norm_w, void *y,
                                         const gd_hip_linear_params *params, int big_tiles, int vector_store,
                                         int compute_units)
{
    const gd_hip_linear_params p = gd_tile_streamed(*params);
    const uint32_t units = ((uint32_t)(compute_units > 0 ? compute_units : 256) + 7u) & ~7u;
    const gd_elem *xp = (const gd_elem *)x, *rp = (const gd_elem *)residual;
    gd_elem *yp = (gd_elem *)y;
    const int e = GD_LINEAR_FN(gd_hip_try_launch_linear_tile_nk)(stream, x, w, bias, residual, y, &p, vector_store, units);
    if (e >= 0) return e;
    if (big_tiles) {
        /* The persistent workgroups walk whole rounds of 256 x 256 tiles; a last round that fills only part of the
         * compute units costs a full tile time.  When that costs more than it would with small tiles, the rows of
         * the last, partial round are left to a second launch with 128 x 128 tiles (rows are independent; two such
         * workgroups fit a compute unit).  A small tile is priced at 0.35 of a big one (a quarter of the work, less
         * reuse of the staged operands). */
        const uint32_t out_bn = p.swiglu_cols != 0u ? 128u : 256u;
        const uint32_t tiles_m = (p.M + 255u) / 256u, tiles_n = (p.N + out_bn - 1u) / out_bn;
        const uint64_t tiles = (uint64_t)tiles_m * tiles_n, rem = tiles % units;
        const uint32_t head_m = (uint32_t)((tiles - rem) / tiles_n); /* row tiles that fill whole rounds */
        if (rem != 0u && head_m != 0u && head_m < tiles_m) {
            const uint32_t head_rows = head_m * 256u, tail_rows = p.M - head_rows;
            const uint64_t small = (uint64_t)((tail_rows + 127u) / 128u) * ((p.N + out_bn / 2u - 1u) / (out_bn / 2u));
            const double whole = (double)((tiles + units - 1u) / units);
            const double cut = (double)(((uint64_t)head_m * tiles_n + units - 1u) / units) +
                               0.35 * (double)((small + 2u * units - 1u) / (2u * units));
            /* whole row tiles when the output allows it (a ragged row tile would leave the direct staging path and take
             * twice as long as the others of its round): the launch covers the LAST rows, so its first rows, fewer than
             * 128, are rows of the head launch computed once more, to the same bits; that needs an output the residual
             * does not alias */
            const bool apart = rp == nullptr || rp + (size_t)p.M * p.ldr <= yp || yp + (size_t)p.M * p.ldy <= rp;
            if (cut + 0.1 < whole) {
                gd_hip_linear_params head = p, tail = p;
                head.M = head_rows;
                tail.M = tail_rows;
                const int e4 = launch_tile<4, 4>(stream, xp, (const gd_elem *)w, (const gd_elem *)bias, rp, (const gd_elem *)norm_w,
                                                 yp, head, (uint32_t)vector_store, units);
                if (e4 != (int)hipSuccess) return e4;
                uint32_t first = head_rows;
                const uint32_t up = (tail_rows + 127u) / 128u * 128u;
                if (apart && up <= p.M) {
                    first = p.M - up;
                    tail.M = up;
                }
                return launch_tile<2, 2>(stream, xp + (size_t)first * p.ldx, (const gd_elem *)w, (const gd_elem *)bias,
                                         rp != nullptr ? rp + (size_t)first * p.ldr : nullptr, (const gd_elem *)norm_w,
                                         yp + (size_t)first * p.ldy, tail, (uint32_t)vector_store, 2u * units);
            }
        }
        return launch_tile<4, 4>(stream, xp, (const gd_elem *)w, (const gd_elem *)bias, rp, (const gd_elem *)norm_w, yp, p,
                                 (uint32_t)vector_store, units);
    }
    return launch_tile<2, 2>(stream, xp, (const gd_elem *)w, (const gd_elem *)bias, rp, (const gd_elem *)norm_w, yp, p,
                             (uint32_t)vector_store, 2u * units);
}

#endif /* GD_LINEAR_TILE_PART */
