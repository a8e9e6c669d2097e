/*
 * Which rows a workgroup of a packed-prompt attention kernel takes: blocks of consecutive rows of one sequence.
 */
#ifndef GD_OPS_SHARED_HIP_ROW_BLOCKS_H
#define GD_OPS_SHARED_HIP_ROW_BLOCKS_H
#include "hip_device.h"

struct gd_row_block {
    uint32_t seq;   /* sequence */
    int start, end; /* its rows */
    uint32_t block; /* number of the block in it */
};

/* Block number `n` of the sequences cu[0] .. cu[batch] in blocks of `size` rows; false behind the last.  The workgroup's work grows
 * with the block's number (causal attention), and workgroups start in the order of their numbers, so that of up to 64 sequences
 * the longest comes first, each from its last block to its first: a launch then ends with short workgroups instead of long ones,
 * and those that run together still share one sequence's keys in the L2s (the last blocks of all sequences first: four times the
 * reads from beyond them, and nothing gained).  Lane t holds sequence t.  More sequences are taken in their order, 64 at a time
 * across the lanes. */
__device__ __forceinline__ bool gd_find_row_block(const int32_t *__restrict__ cu, uint32_t batch, uint32_t size, uint32_t n,
                                                  gd_row_block *found)
{
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t seen = 0u;
    for (uint32_t b0 = 0u; b0 < batch; b0 += 64u) {
        int s0 = 0, e0 = 0, src;
        if (b0 + lane < batch) {
            s0 = cu[b0 + lane];
            e0 = cu[b0 + lane + 1u];
        }
        const uint32_t nb = e0 > s0 ? ((uint32_t)(e0 - s0) + size - 1u) / size : 0u;
        if (batch <= 64u) {
            uint32_t blocks = nb; /* of the longest */
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) blocks = max(blocks, (uint32_t)__shfl_xor((int)blocks, off, 64));
            blocks = (uint32_t)__builtin_amdgcn_readfirstlane((int)blocks);
            uint32_t left = (uint32_t)__builtin_amdgcn_readfirstlane((int)n);
            unsigned long long in; /* the sequences of so many blocks */
            for (;; --blocks) {
                if (blocks == 0u) return false;
                in = __builtin_amdgcn_ballot_w64(nb == blocks);
                const uint32_t here = (uint32_t)__builtin_popcountll(in) * blocks;
                if (left < here) break;
                left -= here;
            }
            for (; left >= blocks; left -= blocks) in &= in - 1ull;
            src = __builtin_ctzll(in);
            found->block = blocks - 1u - left;
        } else {
            uint32_t incl = nb; /* inclusive sum over the lanes below and this one */
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const uint32_t up = (uint32_t)__shfl_up((int)incl, off, 64);
                if ((int)lane >= off) incl += up;
            }
            const unsigned long long hit = __builtin_amdgcn_ballot_w64(seen + incl > n);
            if (hit == 0ull) {
                seen += (uint32_t)__shfl((int)incl, 63, 64);
                continue;
            }
            src = __builtin_ctzll(hit);
            found->block = n - (seen + (uint32_t)__shfl((int)(incl - nb), src, 64));
        }
        found->block = (uint32_t)__builtin_amdgcn_readfirstlane((int)found->block);
        found->seq = (uint32_t)__builtin_amdgcn_readfirstlane((int)b0 + src);
        found->start = __builtin_amdgcn_readfirstlane(__shfl(s0, src, 64));
        found->end = __builtin_amdgcn_readfirstlane(__shfl(e0, src, 64));
        return true;
    }
    return false;
}

/* Sequence number `n` by length, the longest first (of up to 64; of more, n itself), for workgroups that each take a whole sequence:
 * lane t holds sequence t and counts those in front of it. */
__device__ __forceinline__ uint32_t gd_sequence_by_length(const int32_t *__restrict__ cu, uint32_t batch, uint32_t n)
{
    if (batch > 64u || n >= batch) return n;
    const uint32_t lane = threadIdx.x & 63u;
    const int rows = lane < batch ? cu[lane + 1u] - cu[lane] : 0;
    uint32_t rank = 0u;
    for (uint32_t t = 0u; t < batch; ++t) {
        const int other = __builtin_amdgcn_readlane(rows, (int)t);
        rank += other > rows || (other == rows && t < lane) ? 1u : 0u;
    }
    return (uint32_t)__builtin_ctzll(__builtin_amdgcn_ballot_w64(lane < batch && rank == n));
}

#endif
