/* Operands that the many-row projections over [N,K] weights (linear_tile_nk.hip) take beside a matrix. */
#ifndef GD_LINEAR_TILE_NK_H
#define GD_LINEAR_TILE_NK_H
#include "linear_elem.h"

/* Rotation + cache append epilogue of the packed prefill's qkv projection: rotated q rows go to q [M, hd], rotated k rows
 * and v rows into cache row cache_row[m] of the K / V caches (row pitch hd), and there is no [M, 3 hd] intermediate.
 * cos / sin hold, F32, the angles of row m's position for the half_d pairs of a head (NeoX pairing: column c of a head with
 * column c + half_d) in the layout of the table kernel (gd_rope_table_at in ops/qkv_split_rope/hip/qkv_split_rope.hip). */
struct gd_tile_rope {
    const float *cos, *sin;
    const int32_t *cache_row; /* [M]; negative: the row's k and v go nowhere */
    gd_elem *q, *k_cache, *v_cache;
    uint32_t hd;     /* heads * head_dim, a multiple of 256 */
    uint32_t half_d; /* 32 or 64 */
};

/* The rows are packed by group (the experts of a routed feed-forward), and every group has its own weights, one behind the
 * other.  tiles [0]: number of row tiles, then from [2] on (group, first row) of each: a tile's rows, or as many as there
 * are up to the group's end first[group + 1]. */
struct gd_tile_group {
    const int32_t *first, *tiles;
    uint32_t w_rows; /* weight rows of a group */
};

/* Streaming stores for outputs larger than the L2s together: what reads a smaller one finds part of it there.  Two projections, a
 * gated one and a normalised residual addition behind them, BF16, us, with ordinary and with streaming stores: 2048 rows of 2048
 * columns (outputs of 17, 23 and 8 MB) 232.5 (247.5), 4096 x 1024 (17, 23, 8) 137.4 (145.1); 16384 x 1024 (67, 92, 34) 470 (457),
 * 16384 x 2048 (134, 185, 67) 1421 (1400).  Where the line lies between, whole prefills with all stores streaming, and streaming
 * beyond 32 and from 64 MiB on: 18,000 rows of a 512-column F16 decoder (outputs of 19 to 57 MB) 2109, 2107, 2122; 12,500 rows
 * 878, 879, 887; the BF16 layers of 2048 columns, 3,500 rows (14 to 60 MB) 3828, 3825, 3810; 13,600 rows of 1024 columns
 * 6734, 6737, 6713; others differ by less.  A reader of a larger output pays: the norms and rotations of 24,000 latent rows 31 ->
 * 36 us. */
#define GD_TILE_STREAM_BYTES (32u << 20)
static inline gd_hip_linear_params gd_tile_streamed(const gd_hip_linear_params &params)
{
    gd_hip_linear_params p = params;
    if ((uint64_t)p.M * p.N * 2u > GD_TILE_STREAM_BYTES) p.flags |= GD_HIP_LINEAR_STREAM_Y;
    return p;
}

#endif
