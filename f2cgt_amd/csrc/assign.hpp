// Nearest-centre labels on the matrix cores (assign.hip), for the entry points of encode.hip and kmeans.hip.
#pragma once

#include "common.hpp"

namespace f2cgt {

bool assign_fits(int64_t n, int64_t k);   // up to 64 dimensions, the centres' operands within the LDS budget
int assign_rows(const float* x, const float* centers, int64_t* lab64, uint8_t* lab8, int64_t m, int n, int k, int metric,
                hipStream_t st);

// Training step of several column slices: rows [slices][m][k] (slice_step floats apart), centres [slices][n][k]; every
// slice whose stop flag is zero gets assign_sums_shares sets of n * k sums and n counters of its rows by label, over the
// rows whose bit in keep is set (null: all), and its word of `arrived` cleared.
bool assign_sums_fits(int64_t slices, int64_t n, int64_t k);
int64_t assign_sums_shares(int64_t m, int64_t slices, int64_t k);
int assign_sums(const float* x, int64_t slice_step, const uint32_t* keep, int64_t keep_words, const float* centers,
                const int32_t* stop, float* sums, uint32_t* arrived, int64_t m, int slices, int n, int k, int metric,
                hipStream_t st);

}  // namespace f2cgt
