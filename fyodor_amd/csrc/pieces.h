// Activations of the fp16 prefill GEMMs: each token's row scaled by one power
// of two s = 2^(14 - E) (2^(E-1) <= max |x| < 2^E over the token) and split
// into two fp16 pieces, x s = hi + lo + e: |e| <= 2^-22 |x s|, or 2^-25
// absolute where lo is subnormal (prefill_f16.hip writes them).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace fy {

// Workspace for np tokens (np a multiple of 32): hi[np][cols], lo[np][cols]
// (fp16; every 8 columns in the order 0 2 1 3 4 6 5 7), bsum[np][cols / 256][2][8] (the sum of x s over
// 32-column block j of each 256-column group, times 2^-5, as two fp16
// pieces: [0][j] hi, [1][j] lo; |sum| < 2^19, so the scaled sum is below the
// fp16 range limit; written when cols % 256 == 0) and inv[np] (1 / s, or
// NaN).
struct Pieces {
    _Float16 *hi, *lo, *bsum;
    float *inv;
};

__host__ __device__ inline Pieces pieces_of(void *ws, int cols, int np)
{
    Pieces p;
    p.hi = (_Float16 *)ws;
    p.lo = p.hi + (size_t)np * cols;
    p.bsum = p.lo + (size_t)np * cols;
    p.inv = (float *)(p.bsum + (size_t)np * (cols / 16));
    return p;
}

// Tiled (prefill_tile.hip; rows of whole 256-column groups): the pieces in blocks of 32 tokens
// x 128 columns ([np / 32][cols / 128][32][128]), the sums as [np / 32]
// [cols / 256][2][32][8]. Block (tokens m .., columns 128 s ..) of a plane,
// and group g's sums of tokens m ...
__host__ __device__ inline _Float16 *tiled_block(_Float16 *plane, int cols, int m, int s)
{
    return plane + ((size_t)(m / 32) * (cols / 128) + s) * 4096;
}

__host__ __device__ inline _Float16 *tiled_sums(_Float16 *bsum, int cols, int m, int g)
{
    return bsum + ((size_t)(m / 32) * (cols / 256) + g) * 512;
}

// Splits batch rows of x (one workgroup per token; cols % 32 == 0), tiled or
// as plain rows.
hipError_t launch_split_x(const float *x, int batch, int cols, const Pieces &p, bool tiled, hipStream_t s);

}  // namespace fy
