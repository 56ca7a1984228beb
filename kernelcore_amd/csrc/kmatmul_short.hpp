// kmatmul_short.hpp -- the short-batch K-quant matmul (kmatmul_short.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace kcamd {

// One weight matrix of a launch: y [ncols][rows]; tile0 is filled in by the launcher.
struct ShortPart {
    const uint8_t* qw;
    float* y;
    int rows, q6, tile0;
};
struct ShortGroup {
    ShortPart p[3];
    int nparts;
};
// Whether a per-256 batch the prefill kernel does not take runs on this kernel (else on column tiles).
bool matmulShortRuns(int k, int ncols);
// The parts times the same per-256 slots (ncols columns of length k), in one launch; bit-identical per
// column to the reference.
int launchMatmulShort(ShortGroup g, const int* xq, int k, int ncols, hipStream_t s);

}  // namespace kcamd
