// llg_moe_group.hpp -- the grouping of a batch's (token, slot) pairs by expert,
// shared by both batch forms of the MoE FFN (llg_moe_gemm.hip,
// llg_moe_split.hip).
#pragma once
#include "llg_common.hpp"

#define MOE_GROUP_THREADS 1024

// Pairs p = t*k + s sorted by expert (order within an expert is not
// significant: each row's result depends only on its own token).
// tiles[i] = (expert, first row, rows), at most bm rows; n_tiles[0] = count.
struct MoeGroupArgs {
    const int32_t *ids;
    int n_pairs, n_exp, bm;
    int32_t *row_pair, *pair_row;
    int4 *tiles;
    int32_t *n_tiles;
};

// One workgroup of MOE_GROUP_THREADS.  A few microseconds whatever the batch,
// so it runs beside the conversion of x (in the workgroups after it) instead
// of before it: one launch less.
__device__ __forceinline__ void moe_group(const MoeGroupArgs &a) {
    __shared__ int cnt[64], off[65], fill[64];
    const int tid = threadIdx.x;
    if (tid < 64) {
        cnt[tid] = 0;
        fill[tid] = 0;
    }
    __syncthreads();
    for (int p = tid; p < a.n_pairs; p += blockDim.x) atomicAdd(&cnt[a.ids[p]], 1);
    __syncthreads();
    if (tid == 0) {
        int o = 0, nt = 0;
        for (int e = 0; e < a.n_exp; e++) {
            off[e] = o;
            // the fewest tiles of at most bm rows (each streams the
            // expert's weights once), their sizes within one of each other
            const int n = (cnt[e] + a.bm - 1) / a.bm;
            for (int i = 0, r = 0; i < n; i++) {
                const int rows = cnt[e] / n + (i < cnt[e] % n ? 1 : 0);
                a.tiles[nt++] = make_int4(e, o + r, rows, 0);
                r += rows;
            }
            o += cnt[e];
        }
        off[a.n_exp] = o;
        *a.n_tiles = nt;
    }
    __syncthreads();
    for (int p = tid; p < a.n_pairs; p += blockDim.x) {
        const int e = a.ids[p];
        const int r = off[e] + atomicAdd(&fill[e], 1);
        a.row_pair[r] = p;
        a.pair_row[p] = r;
    }
}
