/*
 * Row kernels of latent attention (gfx950), any sizes, BF16 and F32:
 *   prepare  per new token: cosines and sines of its position; RMS norm of the query latent; RMS norm of the key/value
 *            latent and rotation of the shared key part, both into the token's cache row
 *   query    per token and head: the unrotated query taken through the key up-projection, so that its product with a
 *            latent is its product with the key (q . (W_uk c) = (W_uk^T q) . c), and the rotated part turned to its
 *            position: one absorbed query row of a cache row's layout
 *   attend   per token and head: softmax over the sequence's cache rows up to the token's own, and the weighted sum of
 *            their latents (scores, weights and sums in F32)
 *   value    per token and head: the value up-projection of that sum, times the sigmoid of the output gate
 * They are the F32 path and the path of sizes outside the matrix-core kernels (latent_decode.hip, latent_prefill.hip).
 * Bound by round trips and by re-reading the up-projections: elements are requested sixteen, outputs four or eight at a time, and
 * four rows share a reading where there are many, with every sum in the order of the plain loop (mean over portions of 160 to 570
 * rows, 8 heads, F32: query 47 -> 24, attend 132 -> 103, value 81 -> 33 us).
 */
#include "../../_shared/hip_device.h"
#include "hip_latent_attention_types.h"

template <typename T>
__global__ void __launch_bounds__(256)
gd_latent_prepare_kernel(const T *__restrict__ proj, uint32_t ld, const float *__restrict__ q_norm,
                         const float *__restrict__ kv_norm, const float *__restrict__ freq, float *__restrict__ angles,
                         T *__restrict__ cq, T *__restrict__ cache, gd_hip_latent_params m, gd_hip_seqs q)
{
    __shared__ float red[2][4];
    const uint32_t row = blockIdx.x;
    const T *pq = proj + (size_t)row * ld, *pc = pq + m.q_rank, *pr = pc + m.kv_rank;
    int32_t s, pos, slot;
    const bool live = gd_seq_of_row(q, row, &s, &pos, &slot) && (uint32_t)pos < m.tmax;
    float sq = 0.f, sc = 0.f;
    for (uint32_t c = threadIdx.x; c < m.q_rank; c += 256u) sq = fmaf((float)pq[c], (float)pq[c], sq);
    for (uint32_t c = threadIdx.x; c < m.kv_rank; c += 256u) sc = fmaf((float)pc[c], (float)pc[c], sc);
    sq = gd_block_sum<4>(sq, red[0]);
    sc = gd_block_sum<4>(sc, red[1]);
    const float iq = 1.0f / sqrtf(sq / (float)m.q_rank + m.eps), ic = 1.0f / sqrtf(sc / (float)m.kv_rank + m.eps);
    for (uint32_t c = threadIdx.x; c < m.q_rank; c += 256u) cq[(size_t)row * m.q_rank + c] = (T)((float)pq[c] * iq * q_norm[c]);
    if (!live) return;
    T *dst = cache + ((size_t)slot * m.tmax + (uint32_t)pos) * m.pitch;
    for (uint32_t c = threadIdx.x; c < m.kv_rank; c += 256u) dst[c] = (T)((float)pc[c] * ic * kv_norm[c]);
    const uint32_t half = m.rot_dim / 2u;
    for (uint32_t i = threadIdx.x; i < half; i += 256u) {
        const float u = (float)pr[i], v = (float)pr[half + i];
        float s1, c1;
        sincosf((float)pos * freq[i], &s1, &c1);
        angles[(size_t)row * m.rot_dim + i] = c1;
        angles[(size_t)row * m.rot_dim + half + i] = s1;
        dst[m.kv_rank + i] = (T)(u * c1 - v * s1);
        dst[m.kv_rank + half + i] = (T)(v * c1 + u * s1);
    }
    for (uint32_t c = m.kv_rank + m.rot_dim + threadIdx.x; c < m.pitch; c += 256u) dst[c] = (T)0.f;
}

/* prepare for BF16 rows of q_rank + kv_rank <= 4096 in 16-byte pieces: a wavefront per row, the row in registers; bound by its
 * round trips, so everything the row needs is requested in front of the sums (64 rows of 512 + 256, a workgroup each: 6.5 -> 5.2
 * us; 24,000 rows: 36 us either way behind a projection that stores past the L2s, 31 behind one that does not) */
__global__ void __launch_bounds__(256)
gd_latent_prepare_vec_kernel(const gd_bf16 *__restrict__ proj, uint32_t ld, const float *__restrict__ q_norm,
                             const float *__restrict__ kv_norm, const float *__restrict__ freq, float *__restrict__ angles,
                             gd_bf16 *__restrict__ cq, gd_bf16 *__restrict__ cache, gd_hip_latent_params m, gd_hip_seqs q)
{
    constexpr int KEEP = 8;
    const uint32_t row = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6), lane = threadIdx.x & 63u;
    if (row >= q.rows) return;
    const gd_bf16 *pr = proj + (size_t)row * ld, *rot = pr + m.q_rank + m.kv_rank;
    const uint32_t qc = m.q_rank / 8u, all = qc + m.kv_rank / 8u, half = m.rot_dim / 2u;
    int32_t s, pos, slot;
    const bool live = gd_seq_of_row(q, row, &s, &pos, &slot) && (uint32_t)pos < m.tmax;
    gd_bf16x8 v[KEEP];
    gd_float4 w[KEEP][2];
    float sq = 0.f, sc = 0.f, r0 = 0.f, r1 = 0.f, f = 0.f;
#pragma unroll
    for (int i = 0; i < KEEP; ++i) {
        const uint32_t c = lane + 64u * i;
        if (c >= all) continue;
        v[i] = *reinterpret_cast<const gd_bf16x8 *>(pr + c * 8u);
        const float *wp = c < qc ? q_norm + c * 8u : kv_norm + (c - qc) * 8u;
        w[i][0] = *reinterpret_cast<const gd_float4 *>(wp);
        w[i][1] = *reinterpret_cast<const gd_float4 *>(wp + 4);
    }
    if (lane < half) {
        r0 = (float)rot[lane];
        r1 = (float)rot[half + lane];
        f = freq[lane];
    }
#pragma unroll
    for (int i = 0; i < KEEP; ++i) {
        const uint32_t c = lane + 64u * i;
        if (c >= all) continue;
        float ss = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) ss = fmaf((float)v[i][e], (float)v[i][e], ss);
        if (c < qc) sq += ss;
        else sc += ss;
    }
    sq = gd_wave_sum(sq);
    sc = gd_wave_sum(sc);
    const float iq = 1.0f / sqrtf(sq / (float)m.q_rank + m.eps), ic = 1.0f / sqrtf(sc / (float)m.kv_rank + m.eps);
    gd_bf16 *dst = cache + ((size_t)(live ? slot : 0) * m.tmax + (uint32_t)(live ? pos : 0)) * m.pitch;
#pragma unroll
    for (int i = 0; i < KEEP; ++i) {
        const uint32_t c = lane + 64u * i;
        if (c >= all) continue;
        const bool is_q = c < qc;
        const float inv = is_q ? iq : ic;
        gd_bf16x8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = (gd_bf16)((float)v[i][e] * inv * w[i][e >> 2][e & 3]);
        if (is_q) *reinterpret_cast<gd_bf16x8 *>(cq + (size_t)row * m.q_rank + c * 8u) = o;
        else if (live) *reinterpret_cast<gd_bf16x8 *>(dst + (c - qc) * 8u) = o;
    }
    if (!live) return;
    for (uint32_t i = lane; i < half; i += 64u) {
        const bool first = i < 64u;
        const float a = first ? r0 : (float)rot[i], b = first ? r1 : (float)rot[half + i];
        float s1, c1;
        sincosf((float)pos * (first ? f : freq[i]), &s1, &c1);
        angles[(size_t)row * m.rot_dim + i] = c1;
        angles[(size_t)row * m.rot_dim + half + i] = s1;
        dst[m.kv_rank + i] = (gd_bf16)(a * c1 - b * s1);
        dst[m.kv_rank + half + i] = (gd_bf16)(b * c1 + a * s1);
    }
    for (uint32_t c = m.kv_rank + m.rot_dim + lane; c < m.pitch; c += 64u) dst[c] = (gd_bf16)0.f;
}

/* R sums of q[i] * w[i] over n elements, ascending, q's rows n floats apart; a thread's own row w in pieces of 16 bytes where it is
 * aligned, sixteen elements requested together */
template <int R, typename T>
__device__ __forceinline__ void gd_latent_row_dot(const float *q, const T *__restrict__ w, uint32_t n, float (&a)[R])
{
    constexpr uint32_t E = 16u / sizeof(T), PIECES = 16u / E;
    typedef T vec __attribute__((ext_vector_type(E)));
    uint32_t i = 0u;
#pragma unroll
    for (int r = 0; r < R; ++r) a[r] = 0.f;
    if ((reinterpret_cast<uintptr_t>(w) & 15u) == 0u) {
        for (; i + 16u <= n; i += 16u) {
            vec v[PIECES];
#pragma unroll
            for (uint32_t p = 0; p < PIECES; ++p) v[p] = *reinterpret_cast<const vec *>(w + i + p * E);
#pragma unroll
            for (uint32_t e = 0; e < 16u; ++e)
#pragma unroll
                for (int r = 0; r < R; ++r) a[r] = fmaf(q[(uint32_t)r * n + i + e], (float)v[e / E][e % E], a[r]);
        }
    }
    for (; i < n; ++i)
#pragma unroll
        for (int r = 0; r < R; ++r) a[r] = fmaf(q[(uint32_t)r * n + i], (float)w[i], a[r]);
}

/* grid (ceil(rows / R), heads); w_ukt [heads, kv_rank, dim]; ql [rows, heads, pitch].  R rows share a reading of the weights */
template <typename T, int R>
__global__ void __launch_bounds__(256)
gd_latent_query_kernel(const T *__restrict__ qv, const T *__restrict__ w_ukt, const float *__restrict__ angles,
                       T *__restrict__ ql, gd_hip_latent_params m, uint32_t rows)
{
    extern __shared__ float sq[]; /* [R][dim] */
    const uint32_t row0 = blockIdx.x * R, h = blockIdx.y, half = m.rot_dim / 2u, n = min(rows - row0, (uint32_t)R);
    for (uint32_t r = 0; r < R; ++r) { /* rows behind the last repeat it */
        const T *src = qv + ((size_t)(row0 + min(r, n - 1u)) * m.heads + h) * (m.dim + m.rot_dim);
        for (uint32_t d = threadIdx.x; d < m.dim; d += 256u) sq[r * m.dim + d] = (float)src[d];
    }
    __syncthreads();
    for (uint32_t c = threadIdx.x; c < m.kv_rank; c += 256u) {
        float a[R];
        gd_latent_row_dot<R>(sq, w_ukt + ((size_t)h * m.kv_rank + c) * m.dim, m.dim, a);
#pragma unroll
        for (uint32_t r = 0; r < R; ++r)
            if (r < n) ql[((size_t)(row0 + r) * m.heads + h) * m.pitch + c] = (T)a[r];
    }
    for (uint32_t r = 0; r < n; ++r) {
        const uint32_t row = row0 + r;
        const T *src = qv + ((size_t)row * m.heads + h) * (m.dim + m.rot_dim);
        T *dst = ql + ((size_t)row * m.heads + h) * m.pitch;
        for (uint32_t i = threadIdx.x; i < half; i += 256u) {
            const float u = (float)src[m.dim + i], v = (float)src[m.dim + half + i];
            const float c1 = angles[(size_t)row * m.rot_dim + i], s1 = angles[(size_t)row * m.rot_dim + half + i];
            dst[m.kv_rank + i] = (T)(u * c1 - v * s1);
            dst[m.kv_rank + half + i] = (T)(v * c1 + u * s1);
        }
        for (uint32_t c = m.kv_rank + m.rot_dim + threadIdx.x; c < m.pitch; c += 256u) dst[c] = (T)0.f;
    }
}

/* Rows row0 .. row0 + R - 1 of one head, which see the first keys, keys + 1, .. rows of a cache slot: a thread per key for the scores,
 * a thread per latent channel for the sums, blocks of 256 keys.  A row's operations and their order do not depend on R; a row that
 * does not see a key of the others leaves it out. */
template <typename T, int R>
__device__ __forceinline__ void gd_latent_attend_rows(const T *__restrict__ ql, const T *__restrict__ rows, float *__restrict__ o_lat,
                                                      const gd_hip_latent_params &m, uint32_t row0, uint32_t h, uint32_t keys,
                                                      float *smem, float (*sp)[256], float (*red)[4])
{
    const uint32_t used = m.kv_rank + m.rot_dim, wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
    float *sq = smem, *so = smem + R * used; /* queries [R][used], sums [R][kv_rank] */
    uint32_t sees[R];
    float mx[R], total[R], keep[R];
    __syncthreads(); /* rows in front of these are done with the memory */
#pragma unroll
    for (uint32_t r = 0; r < R; ++r) {
        const T *src = ql + ((size_t)(row0 + r) * m.heads + h) * m.pitch;
        for (uint32_t c = threadIdx.x; c < used; c += 256u) sq[r * used + c] = (float)src[c];
        for (uint32_t c = threadIdx.x; c < m.kv_rank; c += 256u) so[r * m.kv_rank + c] = 0.f;
        sees[r] = min(keys + r, m.tmax);
        mx[r] = -INFINITY;
        total[r] = 0.f;
    }
    for (uint32_t k0 = 0; k0 < sees[R - 1]; k0 += 256u) {
        __syncthreads();
        const uint32_t k = k0 + threadIdx.x;
        float score[R], p[R];
#pragma unroll
        for (int r = 0; r < R; ++r) score[r] = -INFINITY;
        if (k < sees[R - 1]) {
            float a[R];
            gd_latent_row_dot<R>(sq, rows + (size_t)k * m.pitch, used, a);
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (k < sees[r]) score[r] = a[r] * m.scale;
        }
        /* maximum of the block's scores */
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float t = gd_wave_max(score[r]);
            if (lane == 0u) red[r][wave] = t;
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float t = fmaxf(fmaxf(red[r][0], red[r][1]), fmaxf(red[r][2], red[r][3]));
            const float nmx = fmaxf(mx[r], t);
            keep[r] = expf(mx[r] - nmx);
            p[r] = k < sees[r] ? expf(score[r] - nmx) : 0.f;
            sp[r][threadIdx.x] = p[r];
            mx[r] = nmx;
        }
        __syncthreads(); /* the maxima are read */
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float t = gd_wave_sum(p[r]);
            if (lane == 0u) red[r][wave] = t;
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < R; ++r) {
            float t = 0.f;
#pragma unroll
            for (int w = 0; w < 4; ++w) t += red[r][w];
            total[r] = total[r] * keep[r] + t;
        }
        const uint32_t all = sees[0] > k0 ? min(sees[0] - k0, 256u) : 0u, any = min(sees[R - 1] - k0, 256u); /* keys that every, some row sees */
        for (uint32_t c = threadIdx.x; c < m.kv_rank; c += 256u) {
            float a[R];
#pragma unroll
            for (int r = 0; r < R; ++r) a[r] = so[(uint32_t)r * m.kv_rank + c] * keep[r];
            const T *kr = rows + (size_t)k0 * m.pitch + c;
            uint32_t j = 0;
            for (; j + 16u <= all; j += 16u) { /* sixteen rows requested together */
                float v[16];
#pragma unroll
                for (uint32_t e = 0; e < 16u; ++e) v[e] = (float)kr[(size_t)(j + e) * m.pitch];
#pragma unroll
                for (uint32_t e = 0; e < 16u; ++e)
#pragma unroll
                    for (int r = 0; r < R; ++r) a[r] = fmaf(sp[r][j + e], v[e], a[r]);
            }
            for (; j < any; ++j) {
                const float v = (float)kr[(size_t)j * m.pitch];
#pragma unroll
                for (int r = 0; r < R; ++r) a[r] = k0 + j < sees[r] ? fmaf(sp[r][j], v, a[r]) : a[r];
            }
#pragma unroll
            for (int r = 0; r < R; ++r) so[(uint32_t)r * m.kv_rank + c] = a[r];
        }
    }
#pragma unroll
    for (uint32_t r = 0; r < R; ++r)
        for (uint32_t c = threadIdx.x; c < m.kv_rank; c += 256u)
            o_lat[((size_t)(row0 + r) * m.heads + h) * m.kv_rank + c] = so[r * m.kv_rank + c] / total[r];
}

/* grid (ceil(rows / R), heads); o_lat F32 [rows, heads, kv_rank].  R rows behind each other share a reading of their sequence's cache */
template <typename T, int R>
__global__ void __launch_bounds__(256)
gd_latent_attend_kernel(const T *__restrict__ ql, const T *__restrict__ cache, float *__restrict__ o_lat,
                        gd_hip_latent_params m, gd_hip_seqs q)
{
    extern __shared__ float smem[];
    __shared__ float sp[R][256], red[R][4];
    const uint32_t row0 = blockIdx.x * R, h = blockIdx.y, n = min(q.rows - row0, (uint32_t)R);
    int32_t s[R], pos[R], slot[R];
    bool there[R], together = n == (uint32_t)R;
#pragma unroll
    for (uint32_t r = 0; r < R; ++r) {
        there[r] = r < n && gd_seq_of_row(q, row0 + r, &s[r], &pos[r], &slot[r]);
        together = together && there[r] && s[r] == s[0];
    }
    if (together) {
        gd_latent_attend_rows<T, R>(ql, cache + (size_t)slot[0] * m.tmax * m.pitch, o_lat, m, row0, h, (uint32_t)pos[0] + 1u, smem, sp, red);
        return;
    }
    if constexpr (R > 1) { /* rows of different sequences */
        for (uint32_t r = 0; r < n; ++r) {
            int32_t one, at, place;
            if (!gd_seq_of_row(q, row0 + r, &one, &at, &place)) continue;
            gd_latent_attend_rows<T, 1>(ql, cache + (size_t)place * m.tmax * m.pitch, o_lat, m, row0 + r, h, (uint32_t)at + 1u, smem, sp, red);
        }
    }
}

/* grid (ceil(rows / R), heads); out [rows, heads * vdim].  R rows share a reading of the weights; a wavefront takes every fourth
 * output, OUTS of them at a time: their loads and their exchanges overlap */
template <typename T, int R>
__global__ void __launch_bounds__(256)
gd_latent_value_kernel(const float *__restrict__ o_lat, const T *__restrict__ w_uv, const T *__restrict__ gate,
                       uint32_t ldg, T *__restrict__ out, gd_hip_latent_params m, uint32_t rows)
{
    extern __shared__ float so[]; /* [R][kv_rank] */
    constexpr uint32_t OUTS = R == 1 ? 8u : 4u;
    const uint32_t row0 = blockIdx.x * R, h = blockIdx.y, wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
    const uint32_t n = min(rows - row0, (uint32_t)R);
    for (uint32_t r = 0; r < R; ++r) { /* rows behind the last repeat it */
        const float *src = o_lat + ((size_t)(row0 + min(r, n - 1u)) * m.heads + h) * m.kv_rank;
        for (uint32_t c = threadIdx.x; c < m.kv_rank; c += 256u) so[r * m.kv_rank + c] = src[c];
    }
    __syncthreads();
    for (uint32_t v0 = wave; v0 < m.vdim; v0 += 4u * OUTS) {
        const T *w = w_uv + ((size_t)h * m.vdim + v0) * m.kv_rank;
        float a[OUTS][R];
#pragma unroll
        for (uint32_t i = 0; i < OUTS; ++i)
#pragma unroll
            for (int r = 0; r < R; ++r) a[i][r] = 0.f;
        for (uint32_t c = lane; c < m.kv_rank; c += 64u) {
            float x[OUTS];
#pragma unroll
            for (uint32_t i = 0; i < OUTS; ++i) x[i] = (float)w[(size_t)min(4u * i, m.vdim - 1u - v0) * m.kv_rank + c];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const float o = so[(uint32_t)r * m.kv_rank + c];
#pragma unroll
                for (uint32_t i = 0; i < OUTS; ++i) a[i][r] = fmaf(o, x[i], a[i][r]);
            }
        }
#pragma unroll
        for (uint32_t i = 0; i < OUTS; ++i)
#pragma unroll
            for (int r = 0; r < R; ++r) a[i][r] = gd_wave_sum(a[i][r]);
        /* lane r * OUTS + i stores output i of row r */
        float mine = 0.f;
#pragma unroll
        for (uint32_t i = 0; i < OUTS; ++i)
#pragma unroll
            for (uint32_t r = 0; r < R; ++r)
                if (lane == r * OUTS + i) mine = a[i][r];
        const uint32_t r = lane / OUTS, v = v0 + 4u * (lane % OUTS);
        if (r < n && v < m.vdim) {
            const float g = (float)gate[(size_t)(row0 + r) * ldg + h * m.vdim + v];
            out[(size_t)(row0 + r) * m.heads * m.vdim + h * m.vdim + v] = (T)(mine * gd_sigmoid_f32(g));
        }
    }
}

/* four rows to a workgroup where that leaves two workgroups for every compute unit (six portions of 160 to 570 rows, 8 heads,
 * three of them shared, mean: value 67 -> 33, query 41 -> 24 us), one otherwise, so that every unit has work */
static bool gd_latent_rows_share(uint32_t rows, uint32_t heads, uint32_t units)
{
    return (uint64_t)rows * heads >= 4u * 2u * (uint64_t)units;
}

extern "C" int gd_hip_launch_latent_prepare(hipStream_t stream, const void *proj, uint32_t ld, const float *q_norm,
                                            const float *kv_norm, const float *freq, float *angles, void *cq, void *cache,
                                            const gd_hip_latent_params *m, const gd_hip_seqs *q, int is_f32, int aligned16)
{
    if (!is_f32 && aligned16 && (m->q_rank % 8u) == 0u && (m->kv_rank % 8u) == 0u && m->q_rank + m->kv_rank <= 4096u) {
        /* four rows to a workgroup where there are many, one where there are few (a decode step), so that they spread over the chip */
        const uint32_t per = q->rows >= 1024u ? 4u : 1u;
        gd_latent_prepare_vec_kernel<<<(q->rows + per - 1u) / per, 64u * per, 0, stream>>>(
            (const gd_bf16 *)proj, ld, q_norm, kv_norm, freq, angles, (gd_bf16 *)cq, (gd_bf16 *)cache, *m, *q);
        return (int)hipGetLastError();
    }
#define GD_GO(T) gd_latent_prepare_kernel<T><<<q->rows, 256, 0, stream>>>((const T *)proj, ld, q_norm, kv_norm, freq, angles, (T *)cq, (T *)cache, *m, *q)
    if (is_f32) GD_GO(float); else GD_GO(gd_bf16);
#undef GD_GO
    return (int)hipGetLastError();
}

extern "C" int gd_hip_launch_latent_query(hipStream_t stream, const void *qv, const void *w_ukt, const float *angles,
                                          void *ql, const gd_hip_latent_params *m, const gd_hip_seqs *q, int is_f32,
                                          uint32_t units)
{
#define GD_GO(T, R) gd_latent_query_kernel<T, R><<<dim3((q->rows + R - 1u) / R, m->heads), 256, R * m->dim * sizeof(float), stream>>>((const T *)qv, (const T *)w_ukt, angles, (T *)ql, *m, q->rows)
    if (gd_latent_rows_share(q->rows, m->heads, units) && m->dim <= 2048u) { if (is_f32) GD_GO(float, 4); else GD_GO(gd_bf16, 4); }
    else { if (is_f32) GD_GO(float, 1); else GD_GO(gd_bf16, 1); }
#undef GD_GO
    return (int)hipGetLastError();
}

/* Rows that share a reading of the cache: as above, and where sequences have many rows (a group that lies in two sequences goes row by
 * row), and LDS enough for four rows.  Six portions of 160 to 570 rows, 8 heads of 256 + 64 channels, mean of the
 * three that share: 103 -> 80 us */
extern "C" int gd_hip_launch_latent_attend(hipStream_t stream, const void *ql, const void *cache, float *o_lat,
                                           const gd_hip_latent_params *m, const gd_hip_seqs *q, int is_f32, uint32_t units)
{
    const size_t lds = (m->pitch + m->kv_rank) * sizeof(float);
    if (q->rows == 0u) return (int)hipSuccess;
    if (lds > 48u * 1024u) return (int)hipErrorInvalidValue;
#define GD_GO(T, R) gd_latent_attend_kernel<T, R><<<dim3((q->rows + R - 1u) / R, m->heads), 256, R * lds, stream>>>((const T *)ql, (const T *)cache, o_lat, *m, *q)
    if (gd_latent_rows_share(q->rows, m->heads, units) && q->rows / 16u >= q->seqs && 4u * lds <= 48u * 1024u) {
        if (is_f32) GD_GO(float, 4); else GD_GO(gd_bf16, 4);
    } else {
        if (is_f32) GD_GO(float, 1); else GD_GO(gd_bf16, 1);
    }
#undef GD_GO
    return (int)hipGetLastError();
}

extern "C" int gd_hip_launch_latent_value(hipStream_t stream, const float *o_lat, const void *w_uv, const void *gate,
                                          uint32_t ldg, void *out, uint32_t rows, const gd_hip_latent_params *m, int is_f32,
                                          uint32_t units)
{
    if (rows == 0u) return (int)hipSuccess;
#define GD_GO(T, R) gd_latent_value_kernel<T, R><<<dim3((rows + R - 1u) / R, m->heads), 256, R * m->kv_rank * sizeof(float), stream>>>(o_lat, (const T *)w_uv, (const T *)gate, ldg, (T *)out, *m, rows)
    if (gd_latent_rows_share(rows, m->heads, units)) { if (is_f32) GD_GO(float, 4); else GD_GO(gd_bf16, 4); }
    else { if (is_f32) GD_GO(float, 1); else GD_GO(gd_bf16, 1); }
#undef GD_GO
    return (int)hipGetLastError();
}
