// dense_walk.h - the records that a thread of k_dense_scatter takes: rounds of
// a grid-stride loop, several records a round, counted from the last record
// down. What ends it is the number of records left, never a position past
// them: the step of a full grid (2^21) divides 2^32, so a position compared
// with a count of more than 2^32 - 2^21 wraps to one below it for ever.
#pragma once
#include <stdint.h>

namespace pyr {

struct DenseWalk {
    uint32_t at, stride, n;  // first position of the round
    bool live;
    __host__ __device__ DenseWalk(uint32_t first, uint32_t threads, uint32_t count)
        : at(first), stride(threads), n(count), live(first < count) {}
    __host__ __device__ bool more() const { return live; }
    __host__ __device__ void next(uint32_t per_round) {
        live = n - at > stride * per_round;
        at += stride * per_round;
    }
    // position u of the round: whether it is a record's, and which
    __host__ __device__ bool has(uint32_t u) const { return n - at > u * stride; }
    __host__ __device__ uint32_t record(uint32_t u) const { return n - 1 - at - u * stride; }
};

}  // namespace pyr
