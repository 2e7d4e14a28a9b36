// Batches of ridge systems and the tile order of the FP64 triangle kernels.
#pragma once

#include <hip/hip_runtime.h>

namespace plm {

// Systems that share a matrix and differ in their ridge parameter: one factor,
// parameter and status word each.
constexpr int kMatBatch = 8;
struct MatBatch {
    double* a[kMatBatch];
    double alpha[kMatBatch];
    int* info;
};

// Tile t of the upper block triangle (bi <= bj) of an nt x nt grid, in 8 x 8
// super-tiles row by row, column by column inside one: consecutive tiles share
// panels, so a run of them given to one XCD reuses its L2.
__device__ __forceinline__ void tri_super_tile(int t, int nt, int& bi, int& bj) {
    int s = 0;
    for (;; s += 8) {
        const int h = min(8, nt - s), cols = max(0, nt - s - 8);
        const int tri = h * (h + 1) / 2;
        if (t < tri) {
            int c = 0;
            while (t >= c + 1) t -= ++c;  // column c holds c + 1 tiles
            bi = s + t, bj = s + c;
            return;
        }
        t -= tri;
        if (t < h * cols) {
            bi = s + t % h, bj = s + 8 + t / h;
            return;
        }
        t -= h * cols;
    }
}

}  // namespace plm
