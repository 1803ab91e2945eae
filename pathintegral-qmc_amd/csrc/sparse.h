// The sparse real-coupling sweep (sparse.hip) as the parallel sweep calls it.
#pragma once

#include "piqmc_internal.h"

namespace piqmc {

// One call, with its device buffers: J_perp and temperatures [S], color
// offsets, packed state [R][2][N] words (32-bit up to 64 slices, else 64-bit).
struct SparseCall {
    const piqmc_problem *pb;
    int R, P, S, M, rpw, block;
    bool chains;               // zero Trotter coupling: slices are independent chains
    uint64_t seed;
    uint32_t rbase, sbase;
    const float *jperp, *temps;
    const int *color_off;
    void *packed;
    double *etrace;
};

size_t sparse_lds(int N, int rpw, int word_bytes, int block);
int sparse_launch(const SparseCall &c, hipStream_t st);
int sparse_upload(piqmc_problem &p, const std::vector<int32_t> &order);
void sparse_free(piqmc_problem &p);

}  // namespace piqmc
