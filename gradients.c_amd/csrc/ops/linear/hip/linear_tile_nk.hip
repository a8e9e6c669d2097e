/*
 * Many rows times [N,K] weights, operands as they lie: the projections of a prefill.
 *
 * Same contract and rounding points as linear_tile.hip, which keeps [K,N] weights, prologues and outputs that
 * 16-byte stores do not fit.  A workgroup of 4 wavefronts (2 x 2) owns 32 TM x 32 TN outputs, a wavefront TM x TN tiles of
 * v_mfma_f32_16x16x32.  That instruction, not 32x32x16, because the chip's power limit decides here: both have the
 * same rate per clock, but on random operands in registers 16x16x32 keeps 1.87 PFLOP/s in F16 and 2.0 in BF16 where
 * 32x32x16 keeps 1.20 and 1.25 (an accumulator element moves once per 32 products instead of once per 16).  The
 * weight fragment is the first operand: lane l holds row l % 16 of a tile and its columns 4 (l / 16) .. + 3.
 *
 * Staging.  K tiles of 64 through two LDS stages, filled by buffer loads that write LDS (8 rows of 128 bytes per
 * instruction); chunk c (16 bytes) of row r sits at c ^ (r >> 1 & 7).  A 16-byte read is served in groups of 16 lanes,
 * 0 to 3, 12 to 15 and 20 to 27 the first of them: rows 0 to 3 and 12 to 15 of one chunk and rows 4 to 11 of the next,
 * which this puts into all 64 banks (with c ^ (r & 7) ^ (r >> 3 & 1), right for fragments of 32 rows, half of the
 * cycles in which the LDS was busy were conflicts).  Rows behind the operand's end are out of the descriptor's range: they cost no
 * traffic, and nothing they give is stored.  Columns behind K get such addresses too, and with them zeros.  So ragged
 * tiles run like whole ones.
 *
 * One wavefront per SIMD, its instruction stream laid out by hand.  A K tile is two steps of 32: step 0 multiplies
 * its first half and reads the fragments of the second, step 1 waits for the next K tile, meets the other wavefronts,
 * and multiplies the second half while it reads the next K tile's first fragments and requests the K tile after that
 * into the stage everybody has left.  The loads are spread over the whole step (requested together they hold up the
 * fragment reads: 8192^3 797 us, spread 758).  The next output tile's K tiles simply follow the last ones of this,
 * so no tile waits for its first operands; the first products of a tile take a zero accumulator instead of cleared
 * registers.
 *
 * Epilogue from registers: v_permlane16_swap joins the 8-byte pieces of neighbouring lane groups into 16-byte chunks,
 * which leave as whole 64-byte row pieces; nothing passes through LDS, so no wavefront waits for another.
 *
 * What bounds it: a K tile of 256 x 256 takes 2280 clocks of which the matrix instructions are 2048, at the 1.8 GHz
 * the power limit leaves; an output tile ends with 2 us of packing and 2.5 us of stores.
 */
#include "../../_shared/hip_device.h"
#include "hip_linear_types.h"
#include "linear_elem.h"
#include "linear_tile_nk.h"
#include "../../qkv_split_rope/hip/rope_device.h"
#include <type_traits>
#include <utility>

typedef int gd_nk_int4 __attribute__((ext_vector_type(4)));
typedef unsigned gd_nk_uint2 __attribute__((ext_vector_type(2)));
typedef unsigned gd_nk_uint4 __attribute__((ext_vector_type(4)));
typedef float gd_nk_float4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) unsigned char gd_nk_lds;

#define GD_NK_RAW_BUFFER 0x00020000 /* descriptor word 3: untyped, no swizzle */

/* Profiling build (make TILE_TIMELINE=1): the first wavefront of every workgroup notes, for its first 32 tiles, the
 * 100 MHz real-time counter at the start of the tile, after the K loop and after the epilogue, and the shader clock
 * ticks the K loop took (their ratio is the clock the chip ran at).  gd_hip_linear_tile_timeline copies the notes of
 * the last launch out; bench.py --probe tile_timeline prints them.  Not part of a normal build. */
#if defined(GD_TILE_TIMELINE) && !GD_LINEAR_IS_BF16
__device__ unsigned long long gd_tile_timeline[256 * 32 * 4];
extern "C" __attribute__((visibility("default"))) int gd_hip_linear_tile_timeline(unsigned long long *host)
{
    return (int)hipMemcpyFromSymbol(host, HIP_SYMBOL(gd_tile_timeline), sizeof(gd_tile_timeline));
}
#define GD_TILE_NOTE(slot, value)                                                                              \
    do {                                                                                                        \
        if (threadIdx.x == 0 && blockIdx.x < 256u && tile / gridDim.x < 32u)                                    \
            gd_tile_timeline[(blockIdx.x * 32u + tile / gridDim.x) * 4u + (slot)] = (value);                    \
    } while (0)
#define GD_TILE_CLOCK() __builtin_amdgcn_s_memtime()
#define GD_TILE_TIME() __builtin_amdgcn_s_memrealtime()
#else
#define GD_TILE_NOTE(slot, value) do { } while (0)
#define GD_TILE_CLOCK() 0ull
#define GD_TILE_TIME() 0ull
#endif

/* f(integral_constant 0) .. f(integral_constant N - 1) */
template <class F, int... V>
__device__ __forceinline__ void gd_nk_each_of(std::integer_sequence<int, V...>, F f)
{
    (f(std::integral_constant<int, V>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void gd_nk_each(F f)
{
    gd_nk_each_of(std::make_integer_sequence<int, N>{}, f);
}

/* 16 bytes per lane straight into LDS: lane l's data lands at lds + IMM + 16 l.  Assembly, because the compiler would
 * wait for all such loads before every LDS read; the kernel waits for them itself. */
template <int IMM>
__device__ __forceinline__ void gd_nk_load_lds(uint32_t lds, uint32_t lane_bytes, gd_nk_int4 descriptor)
{
    asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %3, 0 offen lds"
                 :
                 : "s"(lds), "n"(IMM), "v"(lane_bytes), "s"(descriptor)
                 : "memory", "scc");
}

__device__ __forceinline__ float gd_nk_silu(float z)
{
    const float e = __expf(-fabsf(z));
    /* 1 / (1 + e) with e in (0, 1]: the reciprocal instruction is good to one unit in the last place of F32, and the
     * product is rounded to 16 bits afterwards */
    const float inv = __builtin_amdgcn_rcpf(1.0f + e);
    return z * (z >= 0.0f ? inv : e * inv);
}

#if GD_LINEAR_IS_BF16
__device__ __forceinline__ float gd_nk_gated(float value, float gate, uint32_t flags, const gd_hip_linear_params &p)
{
    if (flags & GD_HIP_LINEAR_CLAMPED_GATE) return gd_lin_clamped_gate(value, gate, p.gate_limit, p.gate_alpha);
    if (flags & GD_HIP_LINEAR_GELU_GATE) {
        const float u = 2.0f * 0.7978845608028654f * (gate + 0.044715f * gate * gate * gate);
        const float e = __expf(-fabsf(u)), inv = __builtin_amdgcn_rcpf(1.0f + e);
        return value * gate * (u >= 0.0f ? inv : e * inv);
    }
    return value * gd_nk_silu(gate);
}
#endif

/* the lane's number, made anew: kept over the K loop it would not fit the registers, and a reload would wait for every
 * load in flight */
__device__ __forceinline__ uint32_t gd_nk_lane()
{
    uint32_t all = 0xffffffffu;
    asm volatile("" : "+s"(all));
    return __builtin_amdgcn_mbcnt_hi(all, __builtin_amdgcn_mbcnt_lo(all, 0u));
}

/* KIND: what becomes of a tile */
enum { GD_NK_PLAIN, GD_NK_GATED, GD_NK_ROPE };

/* TM, TN: 16 x 16 tiles of a wavefront.  GROUPED: rows packed by group (the experts of a routed feed-forward), every
 * group with its own weights; the work list says each row tile's group and first row (gd_tile_group).  MODE: the bias
 * (GD_HIP_EPI_*).  HOW: F16, 1 adds a residual; BF16, the flag of the gate function or of what becomes of an output without
 * a gate.  (Forms that branch in the epilogue instead have the conversion of all sums hoisted above the branch, and
 * spill.) */
template <int TM, int TN, int KIND, uint32_t MODE, uint32_t HOW, bool STREAM, bool GROUPED>
__global__ void __launch_bounds__(256, TM * TN > 16 ? 1 : 2)
gd_linear_tile_nk_kernel(const gd_elem *__restrict__ x, const gd_elem *__restrict__ w, const gd_elem *__restrict__ bias,
                         const gd_elem *residual, gd_elem *y, gd_hip_linear_params p, uint32_t tiles_m,
                         uint32_t tiles_n, std::conditional_t<GROUPED, gd_tile_group, gd_tile_rope> extra)
{
    constexpr uint32_t BM = 32u * TM, BN = 32u * TN;
    constexpr uint32_t OUT_BN = KIND == GD_NK_GATED ? BN / 2u : BN; /* output columns of a tile */
    constexpr uint32_t B_AT = TM * TN > 16 ? 32768u : 16384u;       /* weight rows of a stage */
    constexpr uint32_t STAGE = 2u * B_AT;
    constexpr int NM = TM * TN, NF = TM + TN; /* matrix instructions and fragments of a step; loads of a K tile */
    constexpr int READ_EVERY = NM >= 4 * NF ? 2 : 1, LOAD_EVERY = NM / NF, LOAD_FROM = 1;
    static_assert(LOAD_FROM + (NF - 1) * LOAD_EVERY < NM && (NF - 1) * READ_EVERY < NM, "every read and load has a place in its step");
    extern __shared__ __align__(16) unsigned char gd_nk_smem[];
    gd_nk_lds *const smem = (gd_nk_lds *)gd_nk_smem;

    if constexpr (GROUPED) tiles_m = (uint32_t)__builtin_amdgcn_readfirstlane(extra.tiles[0]);
    const uint32_t total = tiles_m * tiles_n;
    uint32_t tile = blockIdx.x;
    if (tile >= total) return;

    const uint32_t lane = threadIdx.x & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t wm = wave >> 1, wn = wave & 1u;

    /* Order of the tiles: XCD t % 8 takes a contiguous run (one longer in the first total % 8 of them) of an order that
     * walks groups of 8 row tiles column by column, so that the workgroups of an XCD share panels in its L2. */
    uint32_t m0 = 0u, n0 = 0u, rows = 0u, weight_row = 0u; /* origin, rows left, first weight row of the group */
    auto locate = [&](uint32_t t) __attribute__((always_inline)) {
        const uint32_t xcd = t & 7u, pid = xcd * (total >> 3) + min(xcd, total & 7u) + (t >> 3);
        const uint32_t width = 8u * tiles_n;
        const uint32_t first_m = (pid / width) * 8u, in = pid % width;
        const uint32_t high = min(tiles_m - first_m, 8u);
        const uint32_t row_tile = first_m + (high == 8u ? in & 7u : in % high);
        n0 = (high == 8u ? in >> 3 : in / high) * OUT_BN;
        if constexpr (GROUPED) {
            const uint32_t group = (uint32_t)__builtin_amdgcn_readfirstlane(extra.tiles[2u + 2u * row_tile]);
            m0 = (uint32_t)__builtin_amdgcn_readfirstlane(extra.tiles[3u + 2u * row_tile]);
            weight_row = group * extra.w_rows;
            rows = min((uint32_t)__builtin_amdgcn_readfirstlane(extra.first[group + 1u]) - m0, BM);
        } else {
            m0 = row_tile * BM;
            rows = min(p.M - m0, BM);
        }
    };

    /* ---- loads: wavefront w fills rows [w BM/4, (w+1) BM/4) of the activation tile and its share of the weights.  A
     * gated tile holds, per wavefront column, BN/4 value rows and then the gate rows of the same outputs, so that a lane
     * has value and gate of an output in its own accumulators (tiles j and j + TN/2). */
    const uint32_t pitch_x = p.ldx * 2u, pitch_w = p.ldw * 2u; /* bytes */
    const uint32_t chunk = (lane & 7u) ^ (lane >> 4); /* of rows 16 n .. + 7; of the 8 rows behind them chunk ^ 4 */
    const uint32_t row_x = wave * (BM / 4u);
    const uint32_t row_w = KIND == GD_NK_GATED ? (wave & 1u) * p.swiglu_cols + (wave >> 1) * (BN / 4u) : wave * (BN / 4u);
    /* byte offsets of the lane's chunk in every load: in vector registers, because a scalar offset is not part of the
     * range check */
    uint32_t at_x[TM], at_w[TN];
#pragma unroll
    for (uint32_t t = 0; t < (uint32_t)TM; ++t) at_x[t] = (row_x + 8u * t + (lane >> 3)) * pitch_x + (chunk ^ (t & 1u) * 4u) * 16u;
#pragma unroll
    for (uint32_t t = 0; t < (uint32_t)TN; ++t) at_w[t] = (row_w + 8u * t + (lane >> 3)) * pitch_w + (chunk ^ (t & 1u) * 4u) * 16u;
    const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
    uint32_t lds_x = (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds0 + row_x * 128u));
    uint32_t lds_w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds0 + B_AT + wave * (BN / 4u) * 128u));
    uint64_t next_x = 0u, next_w = 0u; /* of the next K tile */
    uint32_t bytes_x = 0u, bytes_w = 0u;
    const uint32_t weight_rows = KIND == GD_NK_GATED ? 2u * p.swiglu_cols : p.N;
    auto describe = [&]() __attribute__((always_inline)) {
        const uint64_t left = (uint64_t)(weight_rows - n0) * pitch_w;
        next_x = (uint64_t)(x + (size_t)m0 * p.ldx);
        next_w = (uint64_t)(w + (size_t)(weight_row + n0) * p.ldw);
        bytes_x = rows * pitch_x;
        bytes_w = (uint32_t)(left < 0x7fffffffull ? left : 0x7fffffffull);
    };
    gd_nk_int4 of_x, of_w;
    of_x[3] = of_w[3] = GD_NK_RAW_BUFFER;
    auto descriptors = [&]() __attribute__((always_inline)) {
        of_x[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)next_x);
        of_x[1] = __builtin_amdgcn_readfirstlane((int)(uint32_t)(next_x >> 32));
        of_x[2] = __builtin_amdgcn_readfirstlane((int)bytes_x);
        of_w[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)next_w);
        of_w[1] = __builtin_amdgcn_readfirstlane((int)(uint32_t)(next_w >> 32));
        of_w[2] = __builtin_amdgcn_readfirstlane((int)bytes_w);
    };
    auto load = [&](auto t) __attribute__((always_inline)) {
        constexpr int T = decltype(t)::value, U = T < TM ? 0 : T - TM;
        if constexpr (T < TM) gd_nk_load_lds<T * 1024>(lds_x, at_x[T < TM ? T : 0], of_x);
        else gd_nk_load_lds<U * 1024>(lds_w, at_w[U], of_w);
    };

    /* ---- fragments: lane l reads chunk l / 16 (+ 4 in the second half of K) of row l % 16 */
    gd_elem8 fa[2][TM], fb[2][TN];
    gd_nk_float4 acc[TM][TN];
    const uint32_t frag = (lane & 15u) * 128u + (((lane >> 4) ^ ((lane >> 1) & 7u)) << 4);
    /* [0]: first half of the next K tile, [1]: second half of this */
    uint32_t from_a[2] = {wm * (TM * 2048u) + frag, wm * (TM * 2048u) + (frag ^ 64u)};
    uint32_t from_b[2] = {B_AT + wn * (TN * 2048u) + frag, B_AT + wn * (TN * 2048u) + (frag ^ 64u)};
    auto read = [&](auto half, auto t) __attribute__((always_inline)) {
        constexpr int H = decltype(half)::value, T = decltype(t)::value;
        if constexpr (T < TN) fb[H][T] = *(__attribute__((address_space(3))) gd_elem8 *)(smem + from_b[H] + T * 2048u);
        else fa[H][T - TN] = *(__attribute__((address_space(3))) gd_elem8 *)(smem + from_a[H] + (T - TN) * 2048u);
    };
    using gd_0 = std::integral_constant<int, 0>;
    using gd_1 = std::integral_constant<int, 1>;

    /* prepare: the next K tile's descriptors; flip: the other stage's fragment addresses.  Both sit between matrix
     * instructions: behind a step's last one their scalar instructions would keep the matrix unit waiting. */
    auto step = [&](auto half, auto first, auto prepare, auto flip) __attribute__((always_inline)) {
        constexpr int H = decltype(half)::value;
        constexpr bool FIRST = decltype(first)::value != 0;
        if constexpr (H == 1) {
            __builtin_amdgcn_s_waitcnt(0x0070); /* vmcnt(0) lgkmcnt(0): this wavefront's part of the next K tile is there */
            __builtin_amdgcn_s_barrier();       /* everybody's is, and everybody has read this one */
            asm volatile("" ::: "memory");      /* no read of the compiler's moves up here */
        }
        __builtin_amdgcn_sched_barrier(0);
        gd_nk_each<NM>([&](auto at) __attribute__((always_inline)) {
            constexpr int I = decltype(at)::value, i = I / TN, j = I % TN;
            acc[i][j] = GD_MFMA_16X16X32(fb[H][j], fa[H][i], FIRST ? (gd_nk_float4)(0.f) : acc[i][j]);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (I % READ_EVERY == 0 && I / READ_EVERY < NF)
                read(std::integral_constant<int, H ^ 1>{}, std::integral_constant<int, I / READ_EVERY < NF ? I / READ_EVERY : 0>{});
            constexpr int L = I >= LOAD_FROM && (I - LOAD_FROM) % LOAD_EVERY == 0 ? (I - LOAD_FROM) / LOAD_EVERY : NF;
            if constexpr (H == 1 && L < NF) load(std::integral_constant<int, L < NF ? L : 0>{});
            if constexpr (H == 0 && I == NM / 2 + 2) prepare();
            if constexpr (H == 1 && I == NM / 2 + 2) flip();
            __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (H == 1) __builtin_amdgcn_s_waitcnt(0xC07F); /* lgkmcnt(0): fragments requested half a step ago */
    };

    /* ---- epilogue ---------------------------------------------------------------------------------------------- */
    gd_elem4 bq[TN]; /* bias of the lane's columns */
    int32_t row_to[KIND == GD_NK_ROPE ? TM : 1];
    uint32_t col0 = 0u;   /* first (weight) column of the wavefront; gated: first output column */
    uint32_t region = 0u; /* ROPE: 0 q, 1 k, 2 v */

    /* the four columns of tile (i, j) that this lane holds, rounded with the bias of the mode */
    auto quad = [&](const gd_nk_float4 &a, const gd_elem4 &b) __attribute__((always_inline)) {
        gd_elem4 h;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
#if GD_LINEAR_IS_BF16
            h[r] = (gd_elem)gd_lin_activated(MODE == GD_HIP_EPI_BIAS_F32 ? a[r] + (float)b[r] : a[r], HOW);
#else
            if (MODE == GD_HIP_EPI_NONE) h[r] = (gd_elem)a[r];
            else if (MODE == GD_HIP_EPI_BIAS_F32) h[r] = (gd_elem)(a[r] + (float)b[r]);
            else h[r] = (gd_elem)a[r] + b[r];
#endif
        }
        return h;
    };
    auto quad_gated = [&](const gd_nk_float4 &value, const gd_nk_float4 &gate, const gd_elem4 &bv, const gd_elem4 &bg) __attribute__((always_inline)) {
        gd_elem4 h;
#if GD_LINEAR_IS_BF16
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            constexpr bool biased = MODE == GD_HIP_EPI_BIAS_F32;
            h[r] = (gd_elem)gd_nk_gated(biased ? value[r] + (float)bv[r] : value[r], biased ? gate[r] + (float)bg[r] : gate[r], HOW, p);
        }
#else
        const gd_elem4 hv = quad(value, bv), hg = quad(gate, bg);
#pragma unroll
        for (int r = 0; r < 4; ++r) h[r] = (gd_elem)((float)hv[r] * gd_nk_silu((float)hg[r]));
#endif
        return h;
    };
    /* column tiles a and b of 16 rows: lane l of group g = l / 16 gets 8 consecutive columns, 8 (g / 2) .. of tile a (g
     * even) or b (g odd): groups 1, 3 of the first operand change places with groups 0, 2 of the second */
    auto join = [&](gd_elem4 a, gd_elem4 b) __attribute__((always_inline)) {
        union { gd_elem4 h; uint32_t u[2]; } ua, ub;
        ua.h = a;
        ub.h = b;
        const gd_nk_uint2 s0 = __builtin_amdgcn_permlane16_swap(ua.u[0], ub.u[0], false, false);
        const gd_nk_uint2 s1 = __builtin_amdgcn_permlane16_swap(ua.u[1], ub.u[1], false, false);
        union { uint32_t u[4]; gd_elem8 h; gd_nk_uint4 v; } c;
        c.u[0] = s0[0];
        c.u[1] = s1[0];
        c.u[2] = s0[1];
        c.u[3] = s1[1];
        return c.v;
    };

    /* Stores and residual loads are bounds-checked by their descriptors: rows behind the tile's end have addresses behind
     * the last row, columns behind N get one far out of range. */
    auto finish = [&](uint32_t tm0, uint32_t tn0, uint32_t trows) __attribute__((always_inline)) {
        constexpr bool RES = !GD_LINEAR_IS_BF16 && HOW != 0u;
        constexpr int OUT = KIND == GD_NK_GATED ? TN / 2 : TN; /* output column tiles of a wavefront */
        const uint32_t l = gd_nk_lane();
        const uint32_t in_wave = ((l >> 4) & 1u) * 16u + (l >> 5) * 8u; /* first column of the lane's chunk in a pair of tiles */
        const uint32_t pitch_y = p.ldy * 2u;
        const __amdgpu_buffer_rsrc_t to = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(y + (size_t)tm0 * p.ldy + tn0), 0, (int)(trows * pitch_y), GD_NK_RAW_BUFFER);
        uint32_t at = (wm * (TM * 16u) + (l & 15u)) * pitch_y + (wn * (OUT * 16u) + in_wave) * 2u;
        uint32_t skip[OUT / 2]; /* added to the addresses of the chunks that lie behind column N */
#pragma unroll
        for (int c = 0; c < OUT / 2; ++c) skip[c] = tn0 + wn * (OUT * 16u) + 32u * c + in_wave < p.N ? 0u : 0x80000000u;
        [[maybe_unused]] const uint32_t pitch_r = p.ldr * 2u;
        [[maybe_unused]] const __amdgpu_buffer_rsrc_t from = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(residual + (RES ? (size_t)tm0 * p.ldr + tn0 : 0u)), 0, RES ? (int)(trows * pitch_r) : 0, GD_NK_RAW_BUFFER);
        [[maybe_unused]] uint32_t from_at = (wm * (TM * 16u) + (l & 15u)) * pitch_r + (wn * (OUT * 16u) + in_wave) * 2u;
        /* residual rows two row tiles ahead */
        gd_nk_uint4 res[RES ? 3 : 1][OUT / 2];
        auto request = [&](auto ii) __attribute__((always_inline)) {
            constexpr int i = decltype(ii)::value;
            if constexpr (RES && i < TM) {
#pragma unroll
                for (int c = 0; c < OUT / 2; ++c)
                    res[i % 3][c] = __builtin_amdgcn_raw_buffer_load_b128(from, from_at + skip[c] + 64u * c, 0, 0);
                from_at += 16u * pitch_r;
            }
        };
        request(std::integral_constant<int, 0>{});
        request(std::integral_constant<int, 1>{});
        gd_nk_each<TM>([&](auto ii) __attribute__((always_inline)) {
            constexpr int i = decltype(ii)::value;
            request(std::integral_constant<int, i + 2>{});
            asm volatile("" : "+v"(at));
            gd_nk_uint4 out[OUT / 2];
            gd_nk_each<OUT / 2>([&](auto cc) __attribute__((always_inline)) {
                constexpr int j = 2 * decltype(cc)::value, g = KIND == GD_NK_GATED ? TN / 2 : 0;
                union { gd_nk_uint4 v; gd_elem8 h; } u, r;
                if constexpr (KIND == GD_NK_GATED)
                    u.v = join(quad_gated(acc[i][j], acc[i][j + g], bq[j], bq[j + g]),
                               quad_gated(acc[i][j + 1], acc[i][j + 1 + g], bq[j + 1], bq[j + 1 + g]));
                else u.v = join(quad(acc[i][j], bq[j]), quad(acc[i][j + 1], bq[j + 1]));
                if constexpr (RES) {
                    r.v = res[i % 3][j / 2];
#pragma unroll
                    for (int t = 0; t < 8; ++t) u.h[t] = r.h[t] + u.h[t];
                }
                out[j / 2] = u.v;
            });
#pragma unroll
            for (int c = 0; c < OUT / 2; ++c) __builtin_amdgcn_raw_buffer_store_b128(out[c], to, at + skip[c] + 64u * c, 0, STREAM ? 2 : 0);
            at += 16u * pitch_y;
            __builtin_amdgcn_sched_barrier(0); /* a row tile's conversions at a time: all at once do not fit the registers */
        });
    };

    /* ROPE: the wavefront's 128 columns lie inside q, k or v (hd is a multiple of 256) and hold whole heads, so both
     * columns of a rotation pair (c, c + half_d) are in one lane: tiles j and j + half_d / 16.  The projection is rounded
     * (with its bias), rotated in F32 with the angles of the row's position, rounded again.  A row goes to row m of q or
     * to row cache_row[m] of a cache.  HALF: column tiles of half a head. */
    auto finish_rope = [&](auto half_tag, uint32_t tm0) __attribute__((always_inline)) {
        if constexpr (KIND == GD_NK_ROPE) {
            constexpr int HALF = decltype(half_tag)::value;
            const uint32_t l = gd_nk_lane();
            gd_elem *to = region == 0u ? extra.q : region == 1u ? extra.k_cache : extra.v_cache;
            to += col0 - region * extra.hd + ((l >> 4) & 1u) * 16u + (l >> 5) * 8u;
            const uint32_t first_row = tm0 + wm * (TM * 16u);
            /* tables: blocks of 32 rows, in a block groups of 8 pairs, in a group the low and the high 4 pairs of all rows */
            const int32_t table = (int32_t)((first_row >> 5) * (extra.half_d * 32u) + (l >> 5) * 256u +
                                            ((l >> 4) & 1u) * 128u + (l & 15u) * 4u);
            gd_nk_float4 cs[2][HALF], sn[2][HALF]; /* angles, a row tile ahead */
            auto request = [&](auto ii) __attribute__((always_inline)) {
                constexpr int i = decltype(ii)::value;
                if constexpr (i < TM) {
                    const int32_t a = table + (int32_t)((i / 2) * (extra.half_d * 32u)) + (i & 1) * 64;
#pragma unroll
                    for (int t = 0; t < HALF; ++t) {
                        cs[i % 2][t] = *reinterpret_cast<const gd_nk_float4 *>(extra.cos + (a + 512 * t));
                        sn[i % 2][t] = *reinterpret_cast<const gd_nk_float4 *>(extra.sin + (a + 512 * t));
                    }
                }
            };
            gd_nk_uint4 out[TN / 2];
            auto put = [&](auto ii) __attribute__((always_inline)) {
                constexpr int i = decltype(ii)::value;
                if (row_to[i] < 0) return;
                gd_elem *row = to + (size_t)(uint32_t)row_to[i] * extra.hd;
#pragma unroll
                for (int c = 0; c < TN / 2; ++c) *reinterpret_cast<gd_nk_uint4 *>(row + 32 * c) = out[c];
            };
            if (region < 2u) {
                request(std::integral_constant<int, 0>{});
                gd_nk_each<TM>([&](auto ii) __attribute__((always_inline)) {
                    constexpr int i = decltype(ii)::value;
                    request(std::integral_constant<int, i + 1>{});
                    gd_nk_each<TN / (2 * HALF) * (HALF / 2)>([&](auto uu) __attribute__((always_inline)) {
                        /* head h of the wavefront, tiles t and t + 1 of its halves */
                        constexpr int h = decltype(uu)::value / (HALF / 2), t = 2 * (decltype(uu)::value % (HALF / 2));
                        constexpr int lo = 2 * HALF * h + t, hi = lo + HALF;
                        gd_elem4 a[2], b[2];
#pragma unroll
                        for (int s = 0; s < 2; ++s) {
                            const gd_elem4 u = quad(acc[i][lo + s], bq[lo + s]);
                            const gd_elem4 v = quad(acc[i][hi + s], bq[hi + s]);
#pragma unroll
                            for (int r = 0; r < 4; ++r) {
                                gd_elem c, d;
                                gd_rope_rotate((float)u[r], (float)v[r], cs[i % 2][t + s][r], sn[i % 2][t + s][r], &c, &d);
                                a[s][r] = c;
                                b[s][r] = d;
                            }
                        }
                        out[lo / 2] = join(a[0], a[1]);
                        out[hi / 2] = join(b[0], b[1]);
                    });
                    put(ii);
                    __builtin_amdgcn_sched_barrier(0);
                });
            } else {
                gd_nk_each<TM>([&](auto ii) __attribute__((always_inline)) {
                    constexpr int i = decltype(ii)::value;
                    gd_nk_each<TN / 2>([&](auto cc) __attribute__((always_inline)) {
                        constexpr int j = 2 * decltype(cc)::value;
                        out[j / 2] = join(quad(acc[i][j], bq[j]), quad(acc[i][j + 1], bq[j + 1]));
                    });
                    put(ii);
                    __builtin_amdgcn_sched_barrier(0);
                });
            }
        } else {
            (void)half_tag, (void)tm0;
        }
    };

    /* ---- tiles ------------------------------------------------------------------------------------------------- */
    const uint32_t ktiles = max((p.K + 63u) / 64u, 2u);
    uint32_t kr = 0u; /* K tile of the output tile at m0, n0 that is requested next */
    /* chunks behind K get addresses out of range, and zeros; a second call undoes the first */
    auto cut = [&]() __attribute__((always_inline)) {
        const int32_t left = (int32_t)p.K - (int32_t)(kr * 64u);
        if (left >= 64) return;
        const uint32_t even = (int32_t)(chunk * 8u) < left ? 0u : 0x80000000u, odd = (int32_t)((chunk ^ 4u) * 8u) < left ? 0u : 0x80000000u;
#pragma unroll
        for (int t = 0; t < TM; ++t) at_x[t] ^= (t & 1) ? odd : even;
#pragma unroll
        for (int t = 0; t < TN; ++t) at_w[t] ^= (t & 1) ? odd : even;
    };
    /* from one K tile's requests to the next's: 64 columns on, into the other stage; behind the last K tile the first of
     * the next output tile, or nothing */
    auto prepare = [&]() __attribute__((always_inline)) {
        cut();
        next_x += 128u;
        next_w += 128u;
        lds_x ^= STAGE;
        lds_w ^= STAGE;
        if (++kr == ktiles) {
            kr = 0u;
            if (tile + gridDim.x < total) {
                locate(tile + gridDim.x);
                describe();
            } else {
                bytes_x = bytes_w = 0u;
            }
        }
        cut();
        descriptors();
    };
    auto flip = [&]() __attribute__((always_inline)) {
        from_a[0] ^= STAGE;
        from_a[1] ^= STAGE;
        from_b[0] ^= STAGE;
        from_b[1] ^= STAGE;
    };
    locate(tile);
    describe();
    cut();
    descriptors();
    gd_nk_each<NF>([&](auto t) __attribute__((always_inline)) { load(t); });
    prepare();
    gd_nk_each<NF>([&](auto t) __attribute__((always_inline)) { load(t); });
    __builtin_amdgcn_s_waitcnt(0x0F70 | (NF & 15) | ((NF >> 4) << 14)); /* vmcnt(NF): the first K tile */
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    gd_nk_each<NF>([&](auto t) __attribute__((always_inline)) { read(gd_0{}, t); });
    from_a[0] ^= STAGE;
    from_b[0] ^= STAGE;
    for (;;) {
        const uint32_t tm0 = m0, tn0 = n0, trows = rows;
        /* bias and rows of the epilogue, here so that the wait of the first K tile covers them: in the epilogue they would
         * wait for the next tile's operands */
        if constexpr (MODE != GD_HIP_EPI_NONE) {
            const __amdgpu_buffer_rsrc_t from = __builtin_amdgcn_make_buffer_rsrc((void *)bias, 0, (int)(weight_rows * 2u), GD_NK_RAW_BUFFER);
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const uint32_t c = KIND == GD_NK_GATED ? (j < TN / 2 ? 0u : p.swiglu_cols) + tn0 + wn * (BN / 4u) + (j % (TN / 2)) * 16u
                                                       : tn0 + wn * (BN / 2u) + j * 16u;
                union { gd_nk_uint2 u; gd_elem4 h; } b;
                b.u = __builtin_amdgcn_raw_buffer_load_b64(from, (c + (gd_nk_lane() >> 4) * 4u) * 2u, 0, 0);
                bq[j] = b.h;
            }
        }
        if constexpr (KIND == GD_NK_ROPE) {
            col0 = tn0 + wn * (BN / 2u);
            region = col0 >= 2u * extra.hd ? 2u : (col0 >= extra.hd ? 1u : 0u);
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const uint32_t r = tm0 + wm * (TM * 16u) + 16u * i + (gd_nk_lane() & 15u);
                row_to[i] = region == 0u ? (int32_t)r : extra.cache_row[r];
            }
        }
        [[maybe_unused]] const unsigned long long clock = GD_TILE_CLOCK();
        GD_TILE_NOTE(0, GD_TILE_TIME());
        step(gd_0{}, gd_1{}, prepare, flip);
        step(gd_1{}, gd_0{}, prepare, flip);
        for (uint32_t kt = 1u; kt < ktiles; ++kt) {
            step(gd_0{}, gd_0{}, prepare, flip);
            step(gd_1{}, gd_0{}, prepare, flip);
        }
        GD_TILE_NOTE(1, GD_TILE_TIME());
        GD_TILE_NOTE(3, GD_TILE_CLOCK() - clock);
        if constexpr (KIND == GD_NK_ROPE) {
            if (extra.half_d == 64u) finish_rope(std::integral_constant<int, 4>{}, tm0);
            else finish_rope(std::integral_constant<int, 2>{}, tm0);
        } else {
            finish(tm0, tn0, trows);
        }
        GD_TILE_NOTE(2, GD_TILE_TIME());
        tile += gridDim.x;
        if (tile >= total) break;
    }
    __builtin_amdgcn_s_waitcnt(0x0F70); /* vmcnt(0): no load may write this workgroup's LDS after its end */
}

#ifdef GD_LINEAR_TILE_GROUPED
#define GD_NK_GROUPED true
#define GD_NK_GROUPED_FORMS 1
#else
#define GD_NK_GROUPED false
#define GD_NK_GROUPED_FORMS 0
#endif
using gd_nk_extra = std::conditional_t<GD_NK_GROUPED, gd_tile_group, gd_tile_rope>;

template <int TM, int TN, int KIND, uint32_t MODE, uint32_t HOW, bool STREAM>
static int gd_nk_launch_form(hipStream_t stream, const gd_elem *x, const gd_elem *w, const gd_elem *bias, const gd_elem *residual,
                             gd_elem *y, const gd_hip_linear_params &p, uint32_t tiles_m, uint32_t units, const gd_nk_extra &extra)
{
    constexpr uint32_t OUT_BN = (KIND == GD_NK_GATED ? 16u : 32u) * TN;
    constexpr bool BIG = TM * TN > 16;
    constexpr size_t lds = BIG ? 131072u : 65536u;
    static bool configured = false;
    auto kernel = gd_linear_tile_nk_kernel<TM, TN, KIND, MODE, HOW, STREAM, GD_NK_GROUPED>;
    if (!configured) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return (int)e;
        configured = true;
    }
    const uint32_t tiles_n = (p.N + OUT_BN - 1u) / OUT_BN, places = BIG ? units : 2u * units;
    const uint64_t tiles = (uint64_t)tiles_m * tiles_n;
    /* persistent workgroups: a multiple of 8 keeps the tile -> XCD relation */
    kernel<<<(uint32_t)(tiles < places ? tiles : places), 256, lds, stream>>>(x, w, bias, residual, y, p, tiles_m, tiles_n, extra);
    return (int)hipGetLastError();
}

template <int TM, int TN, int KIND>
static int gd_nk_launch(hipStream_t stream, const gd_elem *x, const gd_elem *w, const gd_elem *bias, const gd_elem *residual,
                        gd_elem *y, const gd_hip_linear_params &p, uint32_t tiles_m, uint32_t units, const gd_nk_extra &extra)
{
    /* streaming stores: an output that asks for them is mostly in 256 x 256 tiles */
    constexpr bool MAY_STREAM = TM == 8 && TN == 8 && KIND != GD_NK_ROPE;
#define GD_GO(MODE, HOW)                                                                                                            \
    do {                                                                                                                            \
        if (MAY_STREAM && (p.flags & GD_HIP_LINEAR_STREAM_Y))                                                                       \
            return gd_nk_launch_form<TM, TN, KIND, MODE, HOW, MAY_STREAM>(stream, x, w, bias, residual, y, p, tiles_m, units, extra); \
        return gd_nk_launch_form<TM, TN, KIND, MODE, HOW, false>(stream, x, w, bias, residual, y, p, tiles_m, units, extra);        \
    } while (0)
#if GD_NK_GROUPED_FORMS
    if constexpr (KIND == GD_NK_GATED) GD_GO(GD_HIP_EPI_NONE, GD_HIP_LINEAR_CLAMPED_GATE);
    else GD_GO(GD_HIP_EPI_NONE, 0u);
#elif GD_LINEAR_IS_BF16
#define GD_MODES(HOW)                                                          \
    do {                                                                       \
        if (p.epilogue == GD_HIP_EPI_BIAS_F32) GD_GO(GD_HIP_EPI_BIAS_F32, HOW); \
        GD_GO(GD_HIP_EPI_NONE, HOW);                                           \
    } while (0)
    if constexpr (KIND == GD_NK_GATED) {
        if (p.flags & GD_HIP_LINEAR_CLAMPED_GATE) GD_MODES(GD_HIP_LINEAR_CLAMPED_GATE);
        if (p.flags & GD_HIP_LINEAR_GELU_GATE) GD_MODES(GD_HIP_LINEAR_GELU_GATE);
    } else if (p.flags & GD_HIP_LINEAR_SQUARE_RELU) {
        GD_MODES(GD_HIP_LINEAR_SQUARE_RELU);
    }
    GD_MODES(0u);
#else
#define GD_MODES(HOW)                                                          \
    do {                                                                       \
        if (p.epilogue == GD_HIP_EPI_BIAS_F32) GD_GO(GD_HIP_EPI_BIAS_F32, HOW); \
        if (p.epilogue == GD_HIP_EPI_BIAS_F16) GD_GO(GD_HIP_EPI_BIAS_F16, HOW); \
        GD_GO(GD_HIP_EPI_NONE, HOW);                                           \
    } while (0)
    if constexpr (KIND == GD_NK_PLAIN) {
        if (p.has_residual) GD_MODES(1u);
    }
    GD_MODES(0u);
#endif
#undef GD_MODES
#undef GD_GO
}

#ifdef GD_LINEAR_TILE_GROUPED
/* y rows packed by group = x rows times the group's weights: p as for gd_hip_launch_linear_tile (M: packed rows; [N,K]
 * weights, N % 8 == 0, K % 8 == 0, 16-byte aligned rows of x, w and y, no bias, no residual); max_tiles: upper bound of the
 * row tiles, of 256 (big_tiles) or 128 rows */
extern "C" int gd_hip_launch_linear_tile_grouped_bf16(hipStream_t stream, const void *x, const void *w, void *y,
                                                      const gd_hip_linear_params *params, const int32_t *first,
                                                      const int32_t *tiles, uint32_t w_rows, uint32_t max_tiles,
                                                      int big_tiles, int compute_units)
{
    const uint32_t units = ((uint32_t)(compute_units > 0 ? compute_units : 256) + 7u) & ~7u;
    const gd_tile_group group = {first, tiles, w_rows};
    const gd_hip_linear_params p = gd_tile_streamed(*params);
    const gd_elem *xp = (const gd_elem *)x, *wp = (const gd_elem *)w;
    gd_elem *yp = (gd_elem *)y;
    /* a lane's byte offsets within a tile's operands are 31-bit numbers */
    if ((uint64_t)(p.swiglu_cols != 0u ? 2u * p.swiglu_cols : 256u) * p.ldw * 2u > 0x7fffffffull || p.ldx > 0x3fffffu || p.ldy > 0x3fffffu)
        return (int)hipErrorInvalidValue;
    if (p.swiglu_cols != 0u) {
        if (big_tiles) return gd_nk_launch<8, 8, GD_NK_GATED>(stream, xp, wp, nullptr, nullptr, yp, p, max_tiles, units, group);
        return gd_nk_launch<4, 4, GD_NK_GATED>(stream, xp, wp, nullptr, nullptr, yp, p, max_tiles, units, group);
    }
    if (big_tiles) return gd_nk_launch<8, 8, GD_NK_PLAIN>(stream, xp, wp, nullptr, nullptr, yp, p, max_tiles, units, group);
    return gd_nk_launch<4, 4, GD_NK_PLAIN>(stream, xp, wp, nullptr, nullptr, yp, p, max_tiles, units, group);
}
#else
/* rows [first, first + rows) in tiles of 32 TM rows */
template <int TM, int TN, int KIND>
static int gd_nk_rows(hipStream_t stream, const gd_elem *x, const gd_elem *w, const gd_elem *bias, const gd_elem *residual,
                      gd_elem *y, const gd_hip_linear_params &p, uint32_t first, uint32_t rows, uint32_t units)
{
    gd_hip_linear_params part = p;
    part.M = rows;
    return gd_nk_launch<TM, TN, KIND>(stream, x + (size_t)first * p.ldx, w, bias,
                                      residual != nullptr ? residual + (size_t)first * p.ldr : nullptr,
                                      y + (size_t)first * p.ldy, part, (rows + 32u * TM - 1u) / (32u * TM), units,
                                      gd_tile_rope{nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 0u, 0u});
}

/* microseconds that a launch of `tiles` tiles takes on `places` places: whole rounds of a time per tile, the last, partly
 * filled one cheaper the longer the launch is (power, not the number of rounds, bounds a long one: 26.8 and 27.3 rounds of
 * 256 x 256 tiles at K = 4096 both take 2.68 ms) */
static double gd_nk_price(uint64_t tiles, uint32_t places, double tile_us)
{
    const uint64_t full = tiles / places;
    const double fill = (double)(tiles % places) / places, least = 1.0 - (double)full / 32.0;
    return tile_us * ((double)full + (fill == 0.0 ? 0.0 : fill > least ? fill : least));
}

/* Tiles of 256 x 256, 192 x 256 or (two to a compute unit) 128 x 128, or whole rounds of the large ones and the remaining rows in
 * smaller ones, whichever the prices make cheapest.  Prices of a tile, fitted to single launches of BF16 products, us for 256, 192
 * and 128 rows: K = 512 17.9, 13.9, 8.5; 2048 46, 37.5, 26; 4096 90, 83, 60; 5632 114, 108, 80.  What they choose (us for the three
 * alone, and large ones with a tail): 9500 x 2048 -> 2048 90, 77 *, 76, 78; 13000 91 *, 108, 101, 92; 20073 142, 146, 143, 136 *;
 * 23402 x 512 -> 1536 54, 42 *, 43, 51; 5000 x 1024 -> 4224 53, 45 *, 48, 50; 2500 x 2048 -> 2048 42, 38, 28 *, 28; 16000 x 5632 -> 2048
 * 249 *, 293, 302, 280; 27000 x 4096 -> 16896 2672 *, 2955, 4085, 2737. */
template <int KIND>
static int gd_nk_split(hipStream_t stream, const gd_elem *x, const gd_elem *w, const gd_elem *bias, const gd_elem *residual,
                       gd_elem *y, const gd_hip_linear_params &p, uint32_t units)
{
    constexpr uint32_t OUT_BN = KIND == GD_NK_GATED ? 128u : 256u; /* output columns of a large tile */
    constexpr double GATE = KIND == GD_NK_GATED ? 1.0 : 0.0, NEVER = 1e30;
    const double kt = (double)((p.K + 63u) / 64u);
    const double large_us = 6.5 + 4.0 * GATE + 1.25 * kt, mid_us = 5.5 + 1.05 * kt, small_us = 2.5 + 2.0 * GATE + 0.8 * kt;
    const uint64_t large_n = (p.N + OUT_BN - 1u) / OUT_BN, small_n = (p.N + OUT_BN / 2u - 1u) / (OUT_BN / 2u);
    auto large = [&](uint32_t rows) { return gd_nk_price((rows + 255u) / 256u * large_n, units, large_us); };
    auto mid = [&](uint32_t rows) { return KIND == GD_NK_PLAIN ? gd_nk_price((rows + 191u) / 192u * large_n, units, mid_us) : NEVER; };
    auto small = [&](uint32_t rows) { return gd_nk_price((rows + 127u) / 128u * small_n, 2u * units, small_us); };
    /* rows of whole rounds of large tiles, and 8 us for a second launch */
    const uint64_t tiles = (p.M + 255u) / 256u * large_n;
    const uint32_t head = (uint32_t)((tiles - tiles % units) / large_n) * 256u;
    uint32_t first = 0u; /* of the rows in mid or small tiles */
    double best = large(p.M);
    bool by_mid = false, all_large = true;
    auto offer = [&](double price, uint32_t from, bool is_mid) {
        if (price >= best) return;
        best = price;
        first = from;
        by_mid = is_mid;
        all_large = false;
    };
    offer(mid(p.M), 0u, true);
    offer(small(p.M), 0u, false);
    if (head != 0u && head < p.M) {
        offer(large(head) + 8.0 + mid(p.M - head), head, true);
        offer(large(head) + 8.0 + small(p.M - head), head, false);
    }
    if (all_large) first = p.M;
    if (first != 0u) {
        const int e = gd_nk_rows<8, 8, KIND>(stream, x, w, bias, residual, y, p, 0u, first, units);
        if (e != (int)hipSuccess || all_large) return e;
    }
    if constexpr (KIND == GD_NK_PLAIN) {
        if (by_mid) return gd_nk_rows<6, 8, KIND>(stream, x, w, bias, residual, y, p, first, p.M - first, units);
    }
    return gd_nk_rows<4, 4, KIND>(stream, x, w, bias, residual, y, p, first, p.M - first, units);
}

/* whether the call is one for the kernel above; vector_store: rows of y and of the residual allow 16-byte accesses */
static bool gd_nk_fits(const gd_hip_linear_params &p, const void *bias, int vector_store)
{
    /* a lane's byte offsets within a tile's operands are 31-bit numbers */
    const uint64_t weight_rows = p.swiglu_cols != 0u ? 2ull * p.swiglu_cols : 256u;
    return p.w_is_nk && p.prologue == GD_HIP_PRO_NONE && vector_store && (p.N % 8u) == 0u && (p.K % 8u) == 0u &&
           ((uintptr_t)bias & 7u) == 0u && p.N < 0x40000000u && weight_rows * p.ldw * 2u <= 0x7fffffffull &&
           p.ldx <= 0x3fffffu && p.ldy <= 0x3fffffu && p.ldr <= 0x3fffffu;
}

/* Returns -1 for a call that is not for this kernel.  Operands as for gd_hip_launch_linear_tile. */
extern "C" int GD_LINEAR_FN(gd_hip_try_launch_linear_tile_nk)(hipStream_t stream, const void *x, const void *w, const void *bias,
                                                const void *residual, void *y, const gd_hip_linear_params *params,
                                                int vector_store, uint32_t units)
{
    if (!gd_nk_fits(*params, bias, vector_store)) return -1;
    return (params->swiglu_cols != 0u ? gd_nk_split<GD_NK_GATED> : gd_nk_split<GD_NK_PLAIN>)(
        stream, (const gd_elem *)x, (const gd_elem *)w, (const gd_elem *)bias, (const gd_elem *)residual, (gd_elem *)y, *params,
        units);
}

#if !GD_LINEAR_IS_BF16
/* The qkv projection of a packed prefill with rotation and cache append in the epilogue (gd_tile_rope): x [M,K],
 * w [3*hd, K], whole 256 x 256 tiles only.  Requires: M % 256 == 0, hd % 256 == 0, K % 64 == 0, K >= 128, 16-byte
 * aligned rows of x, w, q and the caches, half_d 32 or 64 (head size 64 or 128). */
extern "C" int gd_hip_launch_linear_tile_rope(hipStream_t stream, const void *x, const void *w, const void *bias,
                                              const gd_hip_linear_params *params, const float *cos_rows,
                                              const float *sin_rows, const int32_t *cache_row, void *q, void *k_cache,
                                              void *v_cache, uint32_t hd, uint32_t half_d, int compute_units)
{
    const gd_hip_linear_params &p = *params;
    if (p.M == 0u) return (int)hipSuccess;
    if ((p.M % 256u) != 0u || (hd % 256u) != 0u || p.N != 3u * hd || (p.K % 64u) != 0u || p.K < 128u || !p.w_is_nk ||
        p.prologue != GD_HIP_PRO_NONE || p.has_residual || p.swiglu_cols != 0u || (half_d != 32u && half_d != 64u) ||
        ((uintptr_t)bias & 7u) != 0u || p.ldx > 0x3fffffu || p.ldw > 0x3fffffu)
        return (int)hipErrorInvalidValue;
    const uint32_t units = ((uint32_t)(compute_units > 0 ? compute_units : 256) + 7u) & ~7u;
    return gd_nk_launch<8, 8, GD_NK_ROPE>(stream, (const gd_elem *)x, (const gd_elem *)w, (const gd_elem *)bias, nullptr, nullptr,
                                          p, p.M / 256u, units,
                                          gd_tile_rope{cos_rows, sin_rows, cache_row, (gd_elem *)q, (gd_elem *)k_cache,
                                                       (gd_elem *)v_cache, hd, half_d});
}

/* Row tiles of 256 that fill whole rounds of `units` workgroups for an [M, N] output in 256-column tiles: the rows
 * the rope form takes; the rest (a partly filled last round, a ragged last row tile) goes through the plain
 * projection and the table-driven rotation kernel. */
extern "C" uint32_t gd_hip_linear_tile_rope_head_rows(uint32_t M, uint32_t N, int compute_units)
{
    const uint32_t units = ((uint32_t)(compute_units > 0 ? compute_units : 256) + 7u) & ~7u;
    const uint32_t tiles_n = (N + 255u) / 256u, whole_m = M / 256u;
    const uint64_t tiles = (uint64_t)whole_m * tiles_n;
    const uint64_t rounds = tiles / units;
    uint32_t head_m = rounds != 0u ? (uint32_t)(rounds * units / tiles_n) : 0u;
    /* a few tiles beyond whole rounds cost less than they would in small tiles only when the remainder is nearly a
     * round itself */
    if (tiles - (uint64_t)head_m * tiles_n >= (uint64_t)units * 3u / 4u) head_m = whole_m;
    return head_m * 256u;
}
#endif
#endif
