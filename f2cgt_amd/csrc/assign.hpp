// Nearest-centre labels on the matrix cores (assign.hip), for the entry points of encode.hip.
#pragma once

#include "common.hpp"

namespace f2cgt {

bool assign_fits(int64_t n, int64_t k);   // up to 64 dimensions, the centres' operands within the LDS budget
int assign_rows(const float* x, const float* centers, int64_t* lab64, uint8_t* lab8, int64_t m, int n, int k, int metric,
                hipStream_t st);

}  // namespace f2cgt
