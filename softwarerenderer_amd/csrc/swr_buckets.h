// swr_buckets.h — how the binning sort deals tile ids to its 256 buckets.
//
// A bucket is one workgroup's share of the sort, and tiles that hold pairs lie together on the
// screen: in a column, a row, a block.  Ids count row by row, so by the low 8 bits alone a column
// of a target 256 tiles wide (2048 pixels in tiles of 8) is one bucket's, and a column of one
// 240 tiles wide that of 16.  So each run of 256 ids is rotated over the buckets by a Fibonacci
// hash of its number: a bijection of the run onto the buckets, with the id's bits above the low 8
// the tile's number inside its bucket.  Over targets 16 to 1024 tiles wide, the fullest bucket of a
// column, strip, diagonal or block of tiles holds 12 times its share at most (2 on average), 256
// times by the low bits; constant steps from run to run meet widths and slopes at which it holds
// 16 to 255 times its share.  300,000 triangles in a column of 8 pixels of a 2048x2048 target:
// 805 us a draw by the low bits, 588 us with digit passes instead of buckets, 438 us so; in 64
// columns of pixels 252, 248 and 199 us; draws spread over the screen take the same either way.
#pragma once

#include <stdint.h>

namespace swr {

// Buckets that run `high` of 256 tiles is rotated by.
__host__ __device__ inline uint32_t bucket_turn(uint32_t high)
{
    return (high * 0x9E3779B1u) >> 24;
}

// The digit a sort pass goes by: 8 bits of the id from `shift` on, or the id's bucket.
struct TileDigit {
    int shift;
    bool bucket;
    __host__ __device__ uint32_t of(uint32_t tile) const
    {
        return (bucket ? tile + bucket_turn(tile >> 8) : tile >> shift) & 255u;
    }
};

// The tile of a bucket with the bits `high` above the low 8.
__host__ __device__ inline uint32_t bucket_tile(uint32_t bucket, uint32_t high)
{
    return high << 8 | ((bucket - bucket_turn(high)) & 255u);
}

}  // namespace swr
