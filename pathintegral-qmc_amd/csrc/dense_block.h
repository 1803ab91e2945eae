// The blocked dense sweep (dense_block.hip) as the parallel sweep and the
// batch call it.
#pragma once

#include "piqmc_internal.h"

namespace piqmc {

constexpr int kBlockMaxN = 256;  // spins (four per lane of a wavefront)

// One call's or job's replicas; packed state [R][2][N] words, 32-bit up to 64
// slices, else 64-bit.
struct BlockArgs {
    int N, P, W, S, M, R;
    uint32_t key0, key1, replica_base, sweep_base;
    const float *jperp, *temps;  // [S]
    const int32_t *order;        // [N]
    const float *j2;             // [N][64][slots] twice the couplings by color position (slots = ceil(N / 64))
    const float *jb2;            // [blocks][16][16] those within blocks of 16 positions
    const double *diag;          // [64 * slots] fields by color position
    float bound;                 // at least every row's sum of |J|, fields included
    void *packed;
    double *etrace;              // [R][S] or null
};

// Whether the blocked sweep runs problem p (its tables exist).
inline bool block_applies(const piqmc_problem *p) { return p->d_block != nullptr; }
BlockArgs block_args(const piqmc_problem *p);  // N and the problem's tables filled in
int block_launch(const BlockArgs &a, hipStream_t st);
// Batches: LDS of a job's replica, and the persistent launch over items (job,
// replica) on device arrays.
size_t block_item_lds(const BlockArgs &a);
int block_batch_prepare(size_t lds);
void block_batch_launch(const BlockArgs *jobs, const int2 *items, int n, int *head, int grid, size_t lds, hipStream_t st);
int block_upload(piqmc_problem &p, const std::vector<int32_t> &order);

}  // namespace piqmc
