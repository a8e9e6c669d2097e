/*
 * Projections over F32 operands in true 32-bit arithmetic (F32 matrix instructions or fused multiply-adds, no
 * reduced-precision mode): y = x w^T [+ bias], optionally gated, [N,K] weights.
 *   gd_linear_f32_mfma_kernel  K % 32 == 0 and 16-byte aligned rows: what models call
 *   gd_linear_f32_kernel       any shape, any 4-byte aligned pitch: a 64 x 64 output tile per workgroup of 256 threads,
 *                              4 x 4 outputs per thread, K in LDS tiles of 16
 */
#include "../../_shared/hip_device.h"
#include "hip_linear_types.h"

#define GD_F32_TILE 64
#define GD_F32_BK 16

/* output column n from its sums (v; GATED: g, the gate's); the accurate functions: this path is held to 32-bit rounding */
template <bool GATED>
__device__ __forceinline__ float gd_f32_output(float v, float g, const float *__restrict__ bias, uint32_t n,
                                               const gd_hip_linear_params &p)
{
    if (p.epilogue != GD_HIP_EPI_NONE) v += bias[n];
    if (GATED) {
        if (p.epilogue != GD_HIP_EPI_NONE) g += bias[p.swiglu_cols + n];
        if (p.flags & GD_HIP_LINEAR_CLAMPED_GATE) {
            const float c = fminf(g, p.gate_limit);
            return c / (1.0f + expf(-p.gate_alpha * c)) * (fminf(fmaxf(v, -p.gate_limit), p.gate_limit) + 1.0f);
        }
        if (p.flags & GD_HIP_LINEAR_GELU_GATE)
            return v * (0.5f * g * (1.0f + tanhf(0.7978845608028654f * (g + 0.044715f * g * g * g))));
        return v * (g / (1.0f + expf(-g)));
    }
    if (p.flags & GD_HIP_LINEAR_SQUARE_RELU) return v > 0.f ? v * v : 0.f;
    return v;
}

/* GATED: w has 2 * swiglu_cols rows, the gate of output column n in row swiglu_cols + n */
template <bool GATED>
__global__ void __launch_bounds__(256)
gd_linear_f32_kernel(const float *__restrict__ x, const float *__restrict__ w, const float *__restrict__ bias,
                     float *__restrict__ y, gd_hip_linear_params p)
{
    __shared__ float sx[GD_F32_BK][GD_F32_TILE + 4], sw[GATED ? 2 : 1][GD_F32_BK][GD_F32_TILE + 4];
    const uint32_t m0 = blockIdx.y * GD_F32_TILE, n0 = blockIdx.x * GD_F32_TILE;
    const uint32_t tx = threadIdx.x & 15u, ty = threadIdx.x >> 4;
    float acc[GATED ? 2 : 1][4][4] = {};
    for (uint32_t k0 = 0; k0 < p.K; k0 += GD_F32_BK) {
        for (uint32_t i = threadIdx.x; i < GD_F32_TILE * GD_F32_BK; i += 256u) {
            const uint32_t r = i / GD_F32_BK, k = i % GD_F32_BK;
            const bool kok = k0 + k < p.K, nok = kok && n0 + r < p.N;
            sx[k][r] = kok && m0 + r < p.M ? x[(size_t)(m0 + r) * p.ldx + k0 + k] : 0.f;
            sw[0][k][r] = nok ? w[(size_t)(n0 + r) * p.ldw + k0 + k] : 0.f;
            if (GATED) sw[GATED ? 1 : 0][k][r] = nok ? w[(size_t)(p.swiglu_cols + n0 + r) * p.ldw + k0 + k] : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (uint32_t k = 0; k < GD_F32_BK; ++k) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float a = sx[k][ty + 16u * i];
#pragma unroll
                for (int g = 0; g < (GATED ? 2 : 1); ++g)
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc[g][i][j] = fmaf(a, sw[g][k][tx + 16u * j], acc[g][i][j]);
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t m = m0 + ty + 16u * i, n = n0 + tx + 16u * j;
            if (m >= p.M || n >= p.N) continue;
            const float v = gd_f32_output<GATED>(acc[0][i][j], acc[GATED ? 1 : 0][i][j], bias, n, p);
            y[(size_t)m * p.ldy + n] = v;
        }
    }
}

/*
 * The same on v_mfma_f32_32x32x2_f32 (F32 products and sums).  A wavefront owns a 32 x 32 output tile; operands go from global
 * memory straight into LDS, 8 rows x 128 bytes (32 k) per instruction, and every 16-byte fragment read feeds four matrix
 * instructions: lanes 0-31 hold k 8j .. 8j + 3 of a row and lanes 32-63 the four behind them, for both operands, so
 * instruction i multiplies k 8j + i and 8j + 4 + i.  Chunk c of row r lies at r * 8 + (c ^ (r & 7) ^ ((r >> 3) & 1)): any 16
 * consecutive rows of a chunk hit all 64 banks.
 *   SPLIT false  four wavefronts on a 64 x 64 tile, three LDS stages of 32 k between them, one barrier per stage: bound by the
 *                F32 matrix rate (157 TFLOP/s), operands 16 bytes per clock and compute unit
 *   SPLIT true   all four on one 32 x 32 tile, a quarter of K each, stages of their own and no barrier, summed in wavefront
 *                order at the end: four times as many tiles for outputs that would leave compute units without one, and the
 *                form of few rows, where the weights' bytes decide
 * Both add the same quarters of K in the same order (the first form closes its sums where a quarter ends), so that a row has
 * the same bits whatever rows are beside it: a token replayed alone is the token of the portion.
 * Measured against gd_linear_f32_kernel (us): 6 x 1024 -> 32768 25.9 (151; 5.2 TB/s of weights),
 * 6 x 2816 -> 1024 15.9 (308), 390 x 1024 -> 4384 42 (184; 83 TFLOP/s), 390 x 2816 -> 1024 29 (412), 390 x 1024 -> 2816 gated 74
 * (217; 72 with one running sum), 4096 x 1024 -> 4384 337 (730; 331 with one running sum; 109 TFLOP/s).  Error against 64 bits of a decoder's logits 8e-7 (1.2e-6).
 */
typedef float gd_f32x16 __attribute__((ext_vector_type(16)));

/* lane l's 16 bytes land at lds_base + 16 * l; counted by hand (the compiler would wait for all of them at every LDS read) */
__device__ __forceinline__ void gd_f32_load_lds16(const float *uniform_base, uint32_t lane_byte_offset, uint32_t lds_byte_address)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(lds_byte_address), "v"(lane_byte_offset), "s"(uniform_base)
                 : "memory");
}

template <bool GATED, bool SPLIT>
__global__ void __launch_bounds__(256)
gd_linear_f32_mfma_kernel(const float *__restrict__ x, const float *__restrict__ w, const float *__restrict__ bias,
                          float *__restrict__ y, gd_hip_linear_params p)
{
    constexpr uint32_t TILE = SPLIT ? 32u : 64u;
    constexpr uint32_t STAGES = SPLIT ? 2u : 3u;
    constexpr uint32_t OWNERS = SPLIT ? 4u : 1u;                      /* sets of stages */
    constexpr uint32_t ROWS = TILE * (GATED ? 3u : 2u);               /* x rows, value rows, gate rows of a stage */
    constexpr int ITEMS = (int)(ROWS / 8u / (SPLIT ? 1u : 4u));       /* loads of a wavefront per stage */
    __shared__ __align__(16) unsigned char s_mem[OWNERS * STAGES * ROWS * 128u];
    const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t m0 = blockIdx.y * TILE, n0 = blockIdx.x * TILE;
    const uint32_t blocks = p.K / 32u;
    const uint32_t k_begin = SPLIT ? blocks * wave / 4u : 0u, k_end = SPLIT ? blocks * (wave + 1u) / 4u : blocks;
    const uint32_t own = (SPLIT ? wave : 0u) * (STAGES * ROWS * 128u);
    const uint32_t lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)s_mem + own;

    /* load i of the wavefront: rows 8 * item .. + 7 of the stage; rows behind the last one repeat it and are not stored */
    uint32_t off[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const uint32_t item = SPLIT ? (uint32_t)i : wave * (uint32_t)ITEMS + (uint32_t)i;
        const uint32_t r = item * 8u + lane / 8u, in = r % TILE;
        const uint32_t chunk = (lane & 7u) ^ ((lane >> 3) & 7u) ^ (item & 1u);
        const uint32_t row = r < TILE ? min(m0 + in, p.M - 1u) * p.ldx
                                      : (min(n0 + in, p.N - 1u) + (GATED && r >= 2u * TILE ? p.swiglu_cols : 0u)) * p.ldw;
        off[i] = (row + chunk * 4u) * 4u;
    }
    auto request = [&](uint32_t kb, uint32_t stage) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            const uint32_t item = SPLIT ? (uint32_t)i : wave * (uint32_t)ITEMS + (uint32_t)i;
            gd_f32_load_lds16((item * 8u < TILE ? x : w) + kb * 32u, off[i],
                              __builtin_amdgcn_readfirstlane(lds + (stage * ROWS + item * 8u) * 128u));
        }
    };
    const uint32_t fr = lane & 31u, fh = lane >> 5;
    const uint32_t a_row = (SPLIT ? 0u : (wave >> 1) * 32u) + fr, b_row = TILE + (SPLIT ? 0u : (wave & 1u) * 32u) + fr;
    const uint32_t swizzle = (fr & 7u) ^ ((fr >> 3) & 1u);
    gd_f32x16 acc[GATED ? 2 : 1], sums[GATED ? 2 : 1]; /* of a quarter of K; !SPLIT: of the quarters so far */
#pragma unroll
    for (int g = 0; g < (GATED ? 2 : 1); ++g)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[g][e] = sums[g][e] = 0.f;
    auto multiply = [&](uint32_t stage) __attribute__((always_inline)) {
        const gd_float4 *s = reinterpret_cast<const gd_float4 *>(s_mem + own + stage * (ROWS * 128u));
        gd_float4 a[4], b[GATED ? 2 : 1][4];
#pragma unroll
        for (uint32_t j = 0; j < 4u; ++j) {
            const uint32_t c = (2u * j + fh) ^ swizzle;
            a[j] = s[a_row * 8u + c];
#pragma unroll
            for (uint32_t g = 0; g < (GATED ? 2u : 1u); ++g) b[g][j] = s[(b_row + g * TILE) * 8u + c];
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int g = 0; g < (GATED ? 2 : 1); ++g)
                    acc[g] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[j][e], b[g][j][e], acc[g], 0, 0, 0);
    };
    if (SPLIT) {
        if (k_begin < k_end) request(k_begin, 0u);
        for (uint32_t kb = k_begin; kb < k_end; ++kb) {
            const uint32_t stage = (kb - k_begin) & 1u;
            if (kb + 1u < k_end) {
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); /* the other stage's fragments have been read */
                request(kb + 1u, stage ^ 1u);
                if (GATED) asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
                else asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
            } else {
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            }
            multiply(stage);
        }
    } else {
        request(0u, 0u);
        if (1u < blocks) request(1u, 1u);
        uint32_t stage = 0u, next = 2u;
#pragma unroll 1
        for (uint32_t quarter = 0, kb = 0; quarter < 4u; ++quarter) {
            for (const uint32_t end = blocks * (quarter + 1u) / 4u; kb < end; ++kb) {
                /* this wavefront's loads of block kb have landed once only those of block kb + 1 are outstanding; behind the
                 * barrier everybody's have, and everybody has read block kb - 1, whose stage is filled next */
                if (kb + 1u >= blocks) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
                else if (GATED) asm volatile("s_waitcnt vmcnt(6) lgkmcnt(0)" ::: "memory");
                else asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)" ::: "memory");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                if (kb + 2u < blocks) request(kb + 2u, next);
                multiply(stage);
                stage = stage + 1u == STAGES ? 0u : stage + 1u;
                next = next + 1u == STAGES ? 0u : next + 1u;
            }
#pragma unroll
            for (int g = 0; g < (GATED ? 2 : 1); ++g)
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    sums[g][e] += acc[g][e];
                    acc[g][e] = 0.f;
                }
        }
    }
    static_assert(ITEMS == (SPLIT ? (GATED ? 12 : 8) : (GATED ? 6 : 4)), "the waits above count the loads of a stage");

    /* lane l holds column l % 32 of rows 8 * (r / 4) + 4 * (l / 32) + r % 4 */
    if (!SPLIT) {
        const uint32_t n = n0 + (wave & 1u) * 32u + fr, row0 = m0 + (wave >> 1) * 32u + 4u * fh;
        if (n < p.N) {
#pragma unroll
            for (uint32_t r = 0; r < 16u; ++r) {
                const uint32_t m = row0 + 8u * (r / 4u) + r % 4u;
                if (m < p.M) y[(size_t)m * p.ldy + n] = gd_f32_output<GATED>(sums[0][r], sums[GATED ? 1 : 0][r], bias, n, p);
            }
        }
        return;
    }
    __syncthreads(); /* every wavefront has read its stages: their memory takes the sums */
    float *sum = reinterpret_cast<float *>(s_mem); /* [wave][value, gate][row][column] */
#pragma unroll
    for (uint32_t g = 0; g < (GATED ? 2u : 1u); ++g)
#pragma unroll
        for (uint32_t r = 0; r < 16u; ++r)
            sum[(wave * (GATED ? 2u : 1u) + g) * 1024u + (8u * (r / 4u) + 4u * fh + r % 4u) * 32u + fr] = acc[g][r];
    __syncthreads();
#pragma unroll
    for (uint32_t i = threadIdx.x; i < 1024u; i += 256u) {
        const uint32_t m = m0 + i / 32u, n = n0 + i % 32u;
        float v = 0.f, g = 0.f;
#pragma unroll
        for (uint32_t t = 0; t < 4u; ++t) {
            v += sum[t * (GATED ? 2u : 1u) * 1024u + i];
            if (GATED) g += sum[(t * 2u + 1u) * 1024u + i];
        }
        if (m < p.M && n < p.N) y[(size_t)m * p.ldy + n] = gd_f32_output<GATED>(v, g, bias, n, p);
    }
}

/* compute_units: the tiles of 64 x 64 it takes to fill the chip */
extern "C" int gd_hip_launch_linear_f32(hipStream_t stream, const void *x, const void *w, const void *bias, void *y,
                                        const gd_hip_linear_params *params, int compute_units)
{
    const gd_hip_linear_params &p = *params;
    const float *xp = (const float *)x, *wp = (const float *)w, *bp = (const float *)bias;
    float *yp = (float *)y;
    const bool gated = p.swiglu_cols != 0u;
    if (p.M == 0u || p.N == 0u) return (int)hipSuccess;
    /* whole 128-byte steps of K, 16-byte loads, byte offsets of a row in 31 bits */
    if (p.K != 0u && (p.K % 32u) == 0u && (p.ldx % 4u) == 0u && (p.ldw % 4u) == 0u &&
        (((uintptr_t)x | (uintptr_t)w) & 15u) == 0u && (uint64_t)p.M * p.ldx < (1ull << 29) &&
        ((uint64_t)p.N + p.swiglu_cols) * p.ldw < (1ull << 29) && p.M <= 65535u * 32u) {
        /* 64 x 64 tiles once every compute unit gets one; below that a compute unit without a tile costs more than the
         * second reading of the operands (390 x 2816 -> 1024: 112 large tiles, 416 small ones) */
        const uint64_t big = (uint64_t)((p.M + 63u) / 64u) * ((p.N + 63u) / 64u);
        const bool split = p.M <= 32u || big < (uint64_t)(compute_units > 0 ? compute_units : 256);
        const uint32_t tile = split ? 32u : 64u;
        const dim3 grid((p.N + tile - 1u) / tile, (p.M + tile - 1u) / tile);
#define GD_GO(G, S) gd_linear_f32_mfma_kernel<G, S><<<grid, 256, 0, stream>>>(xp, wp, bp, yp, p)
        if (gated) { if (split) GD_GO(true, true); else GD_GO(true, false); }
        else { if (split) GD_GO(false, true); else GD_GO(false, false); }
#undef GD_GO
        return (int)hipGetLastError();
    }
    const dim3 grid((p.N + GD_F32_TILE - 1u) / GD_F32_TILE, (p.M + GD_F32_TILE - 1u) / GD_F32_TILE);
    if (gated) gd_linear_f32_kernel<true><<<grid, 256, 0, stream>>>(xp, wp, bp, yp, p);
    else gd_linear_f32_kernel<false><<<grid, 256, 0, stream>>>(xp, wp, bp, yp, p);
    return (int)hipGetLastError();
}
