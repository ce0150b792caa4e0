// traceback.h -- tiles and launches of the stochastic traceback.
#pragma once

#include <hip/hip_runtime.h>

#include "engine.h"

namespace aw {

// A traceback tile: columns [c0, c1) of an instance.  The last tile of an
// instance is exact; the chain of another starts from a state sampled from
// column cw alone and walks back to column c1 without storing (a warm-up).
struct Chunk {
    int inst, c0, c1;
    int cw;                  // column where the speculative chain starts (>= c1)
    int first, last;         // first / last tile of its instance
};

// dynamic LDS bytes of the tile kernels for R states per lane
size_t tb_lds_bytes(int R);

// predicted source states of every switch (DevInst::pred); nblk: blocks of
// the batch (blkoff as for the preparation), Rmax: most states per lane
int launch_tb_pred(const DevInst *D, const int *blkoff, int ninst, int nblk, int Rmax,
                   hipStream_t s);

// The chains of the tiles list[0..n): start[j] / end[j] receive the state of
// tile j's chain at column c1 (-1 for an exact tile) and at column c0.
int launch_tb_spec(bool fp32, bool big, const DevInst *D, const Chunk *chunks, const int *list,
                   int n, size_t sh, int *start, int *end, hipStream_t s);

// Re-runs of the tiles idx[0..n) from state k1[x] at their column c1 until
// the samples meet the stored path; res[2x]: that column (-1: none),
// res[2x + 1]: the state at column c0.
int launch_tb_rerun(bool fp32, bool big, const DevInst *D, const Chunk *chunks, const int *idx,
                    const int *k1, int n, size_t sh, int *res, hipStream_t s);

}  // namespace aw
