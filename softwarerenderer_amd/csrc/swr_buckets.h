// swr_buckets.h — how the binning sort deals tile ids to its 256 buckets.
//
// A bucket is one workgroup's share of the sort, and tiles that hold pairs lie together on the
// screen: in a column, a row, a block.  Ids count row by row, so by the low 8 bits alone a column
// of a target 256 tiles wide (2048 pixels in tiles of 8) is one bucket's, and a column of one
// 240 tiles wide that of 16.  So each run of 256 ids is turned by BUCKET_STEP buckets against the
// one before: a bijection of the run onto the buckets, with the id's bits above the low 8 the
// tile's number inside its bucket.  Of the odd steps at which no column, strip, diagonal or block
// of tiles on a target 16 to 1024 tiles wide gives its fullest bucket more than 16 times its share
// (by the low bits 256 times), the step is the one that deals blobs of tiles most evenly: over 1500
// targets with one to three of them the fullest bucket holds 1.32 times the larger of its share
// and the fullest tile, 4.3 times at most (1.75 and 22 by the low bits).  300,000 triangles in a
// column of 8 pixels of a 2048x2048 target: 805 us a draw by the low bits, 588 us with digit passes
// instead of buckets, 440 us so; in 64 columns of pixels 252, 248 and 197 us; draws spread over
// the screen take the same either way.
#pragma once

#include <stdint.h>

namespace swr {

constexpr uint32_t BUCKET_STEP = 165;

// The digit a sort pass goes by: 8 bits of the id from `shift` on, or the id's bucket.
struct TileDigit {
    int shift;
    bool bucket;
    __host__ __device__ uint32_t of(uint32_t tile) const
    {
        return (bucket ? tile + (tile >> 8) * BUCKET_STEP : tile >> shift) & 255u;
    }
};

// The tile of a bucket with the bits `high` above the low 8.
__host__ __device__ inline uint32_t bucket_tile(uint32_t bucket, uint32_t high)
{
    return high << 8 | ((bucket - high * BUCKET_STEP) & 255u);
}

}  // namespace swr
