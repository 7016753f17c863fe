// The sampling points of a problem sorted by the block of base voxels they lie in, and the kernels that work on them
// brick by brick (d2c_brick.hip).
#pragma once
#include "d2c_mma.hpp"

struct BrickDims {
    int nz, nby, nbx;        // base planes -1 .. D-1; blocks of three base voxels along y and x
};
// The block along y or x that base voxel v (-1 on) lies in.  In whole numbers: float quotients go wrong from base voxel 6291457 on, and
// axes reach 2^23.
__host__ __device__ __forceinline__ int brick_block(int v) { return (int)((unsigned)(v + 1) / 3u); }
struct BrickLists {
    int *count;              // points per block
    int *cursor;             // entries given out, then: points outside the volume
    int *end;                // end of a block's entries (they begin `count` before it)
    int *place;              // [n * G + g][tap][p]: a point's entry, -1: no corner inside the volume
    uint4 *pt;               // byte offset of the point's row of 128 bytes (64 channels, float32 32) | its base voxel in the block (y | x << 2); fractions along y, x, z
    float *alpha;            // modulation
};
struct BrickWs {
    size_t count, end, place, pt, alpha, total;     // the sorted points
    size_t res_bytes;                                 // per-point sums of d2c_brick_grad
};
bool d2c_brick_supported(const TiledShape &s, int dtype);
BrickWs d2c_brick_ws(const TiledShape &s);
void *d2c_brick_zero(const TiledShape &s, void *ws, size_t *bytes);
int d2c_brick_sort(const TiledShape &s, const void *off, const void *mask, void *ws, hipStream_t st, bool cleared = false);
int d2c_brick_grad(const TiledShape &s, const void *xcl, const void *gcol, const void *mask, const void *raw, float *gxcl,
                   void *goff, void *gmask, const void *lists, void *res, hipStream_t st);
int d2c_brick_columns(const TiledShape &s, const void *xcl, void *col, int rows, const void *lists, hipStream_t st);
