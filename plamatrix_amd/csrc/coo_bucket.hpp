// COO -> CSR by row ranges: one stable partition of the triplets into buckets of
// whole rows, then one workgroup sorts and folds each bucket in LDS.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "workspace.hpp"

namespace pm
{

constexpr int kBucketCap = 8192;      // triplets a bucket may hold
constexpr int kBucketMean = 3072;     // triplets of an average bucket, at most
constexpr int kBucketMeanLeast = 512; // ... that a smaller conversion is cut down to
constexpr int kBucketsWanted = 256;   // buckets below which the mean shrinks: one per CU
constexpr int kBucketOne = 4608;      // triplets of a conversion that stays one bucket, at most
constexpr int kBucketsMost = 4096;
constexpr int kBucketRowBits = 13;    // a bucket's workgroup also writes its rows' offsets

// How a conversion is cut into buckets; buckets == 0: not by buckets.
struct CooPlan
{
    int buckets = 0;
    int shift = 0;  // row >> shift is the bucket
    int cb = 0;     // bits of a column index; shift + cb <= 32
    int rounds = 0; // triplets per lane of a partition tile
    int64_t tiles = 0;  // 0: one bucket, no partition
};
CooPlan coo_plan(int64_t rows, int64_t cols, int64_t count);

// Bytes behind CooBuckets::tables.
size_t coo_bucket_bytes(const CooPlan& plan);

struct CooBuckets
{
    CooPlan plan;
    int64_t rows, cols, count;
    unsigned long long *keys, *words;  // count each: packed keys, then the sorted (local key, position) words; partitioned words
    char* tables;                      // coo_bucket_bytes
    CooStatus* status;
};

// Partition, sort and count; the status record with the folded nnz goes to `host`
// (pinned) with `ticket`.  When a bucket outgrows kBucketCap or a coordinate is
// out of range, status.unsorted is set and `keys` holds the packed keys.
template <typename S>
int coo_bucket_prepare(const CooBuckets& b, const int64_t* r, const int64_t* c, const S* v, int check_finite,
                       CooStatus* host, unsigned long long ticket, hipStream_t stream);

// Columns, folded values and row offsets from the sorted words; `most`: triplets of
// the largest bucket (the record's).
template <typename S>
int coo_bucket_finish(const CooBuckets& b, const S* v, int check_finite, int64_t capacity, int64_t* row_offsets,
                      int64_t* cols, S* vals, int64_t most, hipStream_t stream);

// What the LSD sort starts from, in `keys` and `positions`: the packed keys and their
// positions in order where the record says unsorted, else the sorted ones.
int coo_bucket_unpack(const CooBuckets& b, unsigned* positions, hipStream_t stream);

} // namespace pm
