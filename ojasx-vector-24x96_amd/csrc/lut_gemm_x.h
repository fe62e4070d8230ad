// lut_gemm_x.h -- where lut_gemm_kernel reads x (no device code, so a host
// check of its bounds needs nothing else).
#pragma once

#include <cstddef>

namespace ojx {

constexpr int kGemmStep = 64;       // input dims per step: four groups of 16

// The kernel stages a step's x in 16-byte units of 8 bf16 values: unit c of
// step s holds dims 64 s + 8 c ...  This is the byte offset of the unit's read
// within a token's row of K values where the rows are not padded; a unit past
// K reads the row's first 16 bytes (K % 16 == 0, so they are there) and is
// zeroed when stored.
constexpr size_t gemm_x_unit(int s, int c, int K) {
    return s * kGemmStep + 8 * c < K ? (size_t)(s * kGemmStep + 8 * c) * 2 : 0;
}

}  // namespace ojx
