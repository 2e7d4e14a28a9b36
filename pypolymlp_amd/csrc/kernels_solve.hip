// FP64 ridge solve on gfx950: blocked Cholesky A = L L^T (panel steps that
// factor, invert and apply a diagonal block in one launch, trailing update on
// FP64 MFMA), triangular solves with the inverses of the diagonal blocks, and
// the residual GEMV used for one step of iterative refinement. Replaces LAPACK
// posv in solver_ridge (src/pypolymlp/mlp_dev/standard/solvers.py:9-84).
//
// Matrices are row-major with leading dimension ld and order n_pad, a multiple
// of 64. Every kernel takes up to kMatBatch systems (one per ridge parameter;
// blockIdx.y), so that the serial parts of one factorization overlap with the
// others'. The factorization reads and writes the lower triangle; the strict
// upper triangle of each 256 x 256 diagonal block receives the transposed
// inverse of that block of L (its diagonal is 1 / L_rr). A factored 64 x 64
// diagonal block waits in a side buffer (n_pad x 64 a system) until the end,
// because the other workgroups of its step read the unfactored one.
#include <hip/hip_runtime.h>

#include "kernels.hpp"
#include "solve_batch.hpp"

namespace plm {

void check_hip(hipError_t e, const char* what);

constexpr int SB = 64;    // panel step and padding granularity
constexpr int NB = 256;   // outer panel, and the diagonal blocks of the solves

typedef __attribute__((__vector_size__(4 * sizeof(double)))) double doublex4;
// a plain vector type: arrays of HIP's double2 class stay in scratch memory
typedef double doublex2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ double read_lane(double v, int lane) {
    union { double d; int i[2]; } u;
    u.d = v;
    u.i[0] = __builtin_amdgcn_readlane(u.i[0], lane);
    u.i[1] = __builtin_amdgcn_readlane(u.i[1], lane);
    return u.d;
}

// sqrt(d) and 1 / sqrt(d) for d > 0: the hardware estimate (about 23 bits) with
// one third-order step of Newton's iteration y' = y (1 + e / 2 + 3 e^2 / 8),
// e = 1 - d y^2, and a last correction of the root
__device__ __forceinline__ void root_and_inverse(double d, double& root, double& inv) {
    if (d > 1e-250 && d < 1e250) {
        double y = __builtin_amdgcn_rsq(d);
        const double e = __builtin_fma(-d * y, y, 1.0);
        y = __builtin_fma(y * e, __builtin_fma(e, 0.375, 0.5), y);
        double r = d * y;
        r = __builtin_fma(__builtin_fma(-r, r, d), 0.5 * y, r);
        root = r, inv = y;
    } else {
        root = sqrt(d), inv = 1.0 / root;
    }
}

// ---------------------------------------------------------------------------
// One 64-column step of a panel, left-looking inside it. Workgroup b owns the
// 64 rows from j0 + 64 b. Every workgroup forms and factors the diagonal block
// itself (64 x 64: cheaper than a second launch), with the columns [k0, j0) of
// the panel subtracted from it and from the workgroup's own rows by MFMA;
// workgroup 0 writes the factor and its inverse, the others their rows times
// L_jj^{-T}, by 16-column blocks with the inverses of the 16 x 16 diagonal
// blocks. Bound by the chain of 64 pivots (about 200 cycles each) and the
// latency of its loads. Before, three launches a step (one-wave factorization
// in LDS, a substitution with one thread per row, an update) took 112 us a
// step at 13,056 rows; this one takes 39 us for two systems.
// ---------------------------------------------------------------------------
constexpr int DP = 66;  // LDS row pitch (doubles) of 64-wide blocks: the 16 rows
                        // x 2 columns of half an operand read hit 64 banks once
constexpr int KC = 32;  // columns of the panel per stage
constexpr int KP = 34;  // their pitch
constexpr int VP = 18;  // pitch of the 16 x 16 inverses
constexpr size_t kStepLds = (size_t)(2 * SB * DP + 4 * 16 * VP + SB) * 8;
static_assert(2 * KP <= 2 * DP, "the stages share the tile's LDS");

// acc += A B^T over 4 s columns: rows ar.. of a (pitch ap), rows br.. of b
__device__ __forceinline__ doublex4 mm16(doublex4 acc, const double* a, int ap, const double* b,
                                         int bp, int steps, int lane) {
    const double* pa = a + (lane & 15) * ap + (lane >> 4);
    const double* pb = b + (lane & 15) * bp + (lane >> 4);
#pragma unroll 4
    for (int s = 0; s < steps; ++s)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(pa[4 * s], pb[4 * s], acc, 0, 0, 0);
    return acc;
}

__global__ void __launch_bounds__(256) chol_step_kernel(MatBatch mb, int ld, int k0, int j0,
                                                        int n, double* __restrict__ side) {
    extern __shared__ __attribute__((aligned(16))) double sm[];
    double* D = sm;                 // the diagonal block, then L_jj
    double* T = D + SB * DP;        // the workgroup's rows; stages before that
    double* V = T + SB * DP;        // inverses of the 16 x 16 diagonal blocks
    double* rinv = V + 4 * 16 * VP; // 1 / L_rr
    double* Pj = T;                 // [64][KC] columns of the panel, rows j0..
    double* Pi = D;                 // rows R0.. (D is written after the stages)
    double* __restrict__ A = mb.a[blockIdx.y];
    int* __restrict__ info = mb.info + blockIdx.y;
    const int R0 = j0 + SB * blockIdx.x;
    const bool diag = blockIdx.x == 0;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wi = (wave >> 1) * 32, wj = (wave & 1) * 32;
    // minus the blocks' elements, to which the products are added: loads without
    // a condition, all in flight while the stages run
    doublex4 ad[2][2], at[2][2];
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int r = wi + 16 * m + (lane >> 4) + 4 * v, c = wj + 16 * q + (lane & 15);
                ad[m][q][v] = -A[(size_t)(j0 + r) * ld + j0 + c];
                at[m][q][v] = -A[(size_t)(R0 + r) * ld + j0 + c];
            }
    // 64 rows x 16 pairs of columns a stage, four pieces a thread
    doublex2 rj[4], ri[4];
    auto load = [&](int kc) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int p = tid + 256 * u, r = p >> 4, c = 2 * (p & 15);
            rj[u] = *reinterpret_cast<const doublex2*>(A + (size_t)(j0 + r) * ld + kc + c);
            ri[u] = *reinterpret_cast<const doublex2*>(A + (size_t)(R0 + r) * ld + kc + c);
        }
    };
    if (k0 < j0) load(k0);
    for (int kc = k0; kc < j0; kc += KC) {
        __syncthreads();
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int p = tid + 256 * u, r = p >> 4, c = 2 * (p & 15);
            *reinterpret_cast<doublex2*>(Pj + r * KP + c) = rj[u];
            *reinterpret_cast<doublex2*>(Pi + r * KP + c) = ri[u];
        }
        __syncthreads();
        if (kc + KC < j0) load(kc + KC);
#pragma unroll
        for (int ks = 0; ks < KC; ks += 4) {
            const int k = ks + (lane >> 4), l = lane & 15;
            double b[2], x[2], y[2];
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                b[m] = Pj[(wj + 16 * m + l) * KP + k];
                x[m] = Pj[(wi + 16 * m + l) * KP + k];
                y[m] = Pi[(wi + 16 * m + l) * KP + k];
            }
#pragma unroll
            for (int m = 0; m < 2; ++m)
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    ad[m][q] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[m], b[q], ad[m][q], 0, 0, 0);
                    at[m][q] = __builtin_amdgcn_mfma_f64_16x16x4f64(y[m], b[q], at[m][q], 0, 0, 0);
                }
        }
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int r = wi + 16 * m + (lane >> 4) + 4 * v, c = wj + 16 * q + (lane & 15);
                D[r * DP + c] = c <= r ? -ad[m][q][v] : 0.0;
                T[r * DP + c] = -at[m][q][v];
            }
    __syncthreads();
    // the diagonal block by 16 columns: one wave factors them on all rows (lane
    // = row, the columns in registers), then the rest of the block is updated
#pragma unroll 1
    for (int b = 0; b < 4; ++b) {
        if (wave == 0) {
            double p[16];
#pragma unroll
            for (int c = 0; c < 16; ++c) p[c] = D[lane * DP + 16 * b + c];
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                double d = read_lane(p[j], 16 * b + j);
                if (!(d > 0.0)) {
                    if (diag && lane == 0 && *info == 0) *info = j0 + 16 * b + j + 1;
                    d = 1.0;  // keep the factor finite; the caller discards this solve
                }
                double root, inv;
                root_and_inverse(d, root, inv);
                if (lane == 0) rinv[16 * b + j] = inv;
                const double l = lane == 16 * b + j ? root : p[j] * inv;
                p[j] = l;
#pragma unroll
                for (int k = j + 1; k < 16; ++k)
                    p[k] = __builtin_fma(-l, read_lane(l, 16 * b + k), p[k]);
            }
#pragma unroll
            for (int c = 0; c < 16; ++c)
                if (lane >= 16 * b + c) D[lane * DP + 16 * b + c] = p[c];
        }
        __syncthreads();
        int t = 0;
        for (int ti = b + 1; ti < 4; ++ti)
            for (int tj = b + 1; tj <= ti; ++tj, ++t) {
                if ((t & 3) != wave) continue;
                const doublex4 s = mm16(doublex4{0, 0, 0, 0}, D + 16 * ti * DP + 16 * b, DP,
                                        D + 16 * tj * DP + 16 * b, DP, 4, lane);
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    D[(16 * ti + (lane >> 4) + 4 * v) * DP + 16 * tj + (lane & 15)] -= s[v];
            }
        __syncthreads();
    }
    // wave w: the inverse of diagonal block w, a column per lane (the upper
    // triangle of the block in D is not read)
    {
        const double* Lw = D + 16 * wave * DP + 16 * wave;
        const int c = lane & 15;
        double x[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            double s = r == c ? 1.0 : 0.0;
#pragma unroll
            for (int k = 0; k < r; ++k) s = __builtin_fma(-Lw[r * DP + k], x[k], s);
            x[r] = s * rinv[16 * wave + r];
        }
        if (lane < 16)
#pragma unroll
            for (int r = 0; r < 16; ++r) V[(16 * wave + r) * VP + c] = r >= c ? x[r] : 0.0;
    }
    __syncthreads();
    if (!diag) {
        // rows 16 wave .. of T: X_c = (T_c - sum_{p < c} X_p L_cp^T) V_c^T
        double* Tw = T + 16 * wave * DP;
#pragma unroll 1
        for (int c = 0; c < 4; ++c) {
            if (c > 0) {
                const doublex4 s = mm16(doublex4{0, 0, 0, 0}, Tw, DP, D + 16 * c * DP, DP, 4 * c, lane);
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    Tw[((lane >> 4) + 4 * v) * DP + 16 * c + (lane & 15)] -= s[v];
            }
            __syncthreads();
            const doublex4 x = mm16(doublex4{0, 0, 0, 0}, Tw + 16 * c, DP, V + 16 * c * VP, VP, 4, lane);
            __syncthreads();
#pragma unroll
            for (int v = 0; v < 4; ++v) Tw[((lane >> 4) + 4 * v) * DP + 16 * c + (lane & 15)] = x[v];
            __syncthreads();
        }
        for (int e = tid; e < SB * SB / 2; e += 256) {
            const int r = e >> 5, c = 2 * (e & 31);
            *reinterpret_cast<doublex2*>(A + (size_t)(R0 + r) * ld + j0 + c) =
                *reinterpret_cast<const doublex2*>(T + r * DP + c);
        }
        return;
    }
    // the inverse of L_jj in T: block (i, j), i > j, is -V_i sum_k L_ik T_kj
    for (int e = tid; e < SB * SB; e += 256) {
        const int r = e >> 6, c = e & 63;
        T[r * DP + c] = (r >> 4) == (c >> 4) ? V[r * VP + (c & 15)] : 0.0;
    }
    __syncthreads();
#pragma unroll 1
    for (int lv = 1; lv < 4; ++lv) {
        const int i = wave, j = wave - lv;
        doublex4 s = {0, 0, 0, 0};
        if (j >= 0) {
            for (int k = j; k < i; ++k)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    s = __builtin_amdgcn_mfma_f64_16x16x4f64(
                        D[(16 * i + (lane & 15)) * DP + 16 * k + 4 * q + (lane >> 4)],
                        T[(16 * k + 4 * q + (lane >> 4)) * DP + 16 * j + (lane & 15)], s, 0, 0, 0);
        }
        __syncthreads();
        if (j >= 0)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                T[(16 * i + (lane >> 4) + 4 * v) * DP + 16 * j + (lane & 15)] = s[v];
        __syncthreads();
        s = doublex4{0, 0, 0, 0};
        if (j >= 0)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                s = __builtin_amdgcn_mfma_f64_16x16x4f64(
                    V[(16 * i + (lane & 15)) * VP + 4 * q + (lane >> 4)],
                    T[(16 * i + 4 * q + (lane >> 4)) * DP + 16 * j + (lane & 15)], s, 0, 0, 0);
        __syncthreads();
        if (j >= 0)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                T[(16 * i + (lane >> 4) + 4 * v) * DP + 16 * j + (lane & 15)] = -s[v];
        __syncthreads();
    }
    side += ((size_t)n * blockIdx.y + j0) * SB;
    for (int e = tid; e < SB * SB; e += 256) {
        const int r = e >> 6, c = e & 63;
        side[e] = c <= r ? D[r * DP + c] : T[c * DP + r];
    }
}

// ---------------------------------------------------------------------------
// The factored 64 x 64 diagonal blocks put in place, and their inverses grown to
// those of the 256 x 256 blocks of L: block (i, j), i > j, of the inverse is -V_i sum_k L_ik W_kj,
// stored transposed at block (j, i). One workgroup per 256-block; 16 products
// of 64^3 each on MFMA.
// ---------------------------------------------------------------------------
constexpr size_t kInvLds = (size_t)2 * SB * DP * 8;

__global__ void __launch_bounds__(256) chol_inverse_kernel(MatBatch mb, int ld, int n,
                                                           const double* __restrict__ side) {
    extern __shared__ __attribute__((aligned(16))) double sm[];
    double* P = sm;
    double* Q = P + SB * DP;
    double* A = mb.a[blockIdx.y];
    const int k0 = blockIdx.x * NB, nb = min(NB, n - k0) / SB;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wi = (wave >> 1) * 32, wj = (wave & 1) * 32;
    side += ((size_t)n * blockIdx.y + k0) * SB;
    for (int e = tid; e < nb * SB * SB; e += 256) {
        const int r = e >> 6, c = (r & ~63) + (e & 63);
        A[(size_t)(k0 + r) * ld + k0 + c] = side[e];
    }
    __threadfence();  // read back below by other threads of this workgroup
    // block (bi, bj) of L, or with inv block (bi, bj) of the inverse
    auto stage = [&](double* dst, int bi, int bj, bool inv) {
        for (int e = tid; e < SB * SB; e += 256) {
            const int r = e >> 6, c = e & 63;
            if (!inv) {
                dst[r * DP + c] = A[(size_t)(k0 + SB * bi + r) * ld + k0 + SB * bj + c];
            } else {
                // element (c, r) of the inverse block is stored at (r, c) of block (bj, bi)
                const double v = A[(size_t)(k0 + SB * bj + r) * ld + k0 + SB * bi + c];
                dst[c * DP + r] = bi != bj || c > r ? v : (c == r ? 1.0 / v : 0.0);
            }
        }
    };
    doublex4 acc[2][2];
    auto clear = [&] {
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int q = 0; q < 2; ++q) acc[m][q] = doublex4{0, 0, 0, 0};
    };
    auto product = [&] {  // acc += P Q
#pragma unroll 4
        for (int ks = 0; ks < SB; ks += 4) {
            const int k = ks + (lane >> 4), l = lane & 15;
            double a[2], b[2];
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                a[m] = P[(wi + 16 * m + l) * DP + k];
                b[m] = Q[k * DP + wj + 16 * m + l];
            }
#pragma unroll
            for (int m = 0; m < 2; ++m)
#pragma unroll
                for (int q = 0; q < 2; ++q)
                    acc[m][q] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[m], b[q], acc[m][q], 0, 0, 0);
        }
    };
    for (int lv = 1; lv < nb; ++lv)
        for (int i = lv; i < nb; ++i) {
            const int j = i - lv;
            clear();
            for (int k = j; k < i; ++k) {
                __syncthreads();
                stage(P, i, k, false);
                stage(Q, k, j, true);
                __syncthreads();
                product();
            }
            __syncthreads();
            stage(P, i, i, true);
#pragma unroll
            for (int m = 0; m < 2; ++m)
#pragma unroll
                for (int q = 0; q < 2; ++q)
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        Q[(wi + 16 * m + (lane >> 4) + 4 * v) * DP + wj + 16 * q + (lane & 15)] =
                            acc[m][q][v];
            __syncthreads();
            clear();
            product();
            __syncthreads();
            // transposed through LDS, so that the stores are in address order
#pragma unroll
            for (int m = 0; m < 2; ++m)
#pragma unroll
                for (int q = 0; q < 2; ++q)
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        P[(wi + 16 * m + (lane >> 4) + 4 * v) * DP + wj + 16 * q + (lane & 15)] =
                            -acc[m][q][v];
            __syncthreads();
            for (int e = tid; e < SB * SB; e += 256) {
                const int r = e >> 6, c = e & 63;
                A[(size_t)(k0 + SB * j + r) * ld + k0 + SB * i + c] = P[c * DP + r];
            }
            __threadfence();  // read back by later products of this workgroup
        }
}

// ---------------------------------------------------------------------------
// Trailing update with a finished panel: C -= P P^T on the lower triangle from
// base on, P = A[base.., k0 : k0 + kw]. 128 x 128 tiles of eight waves (64 x 32
// each, 64 accumulator registers, two workgroups a CU), 16 columns of the panel
// per stage through two LDS buffers, the next stage in registers. A 128-wide
// tile halves the panel traffic of a 64-wide one, which bound it (8 flops a
// byte, 25 TFLOP/s); it runs at 57 TFLOP/s (F = 13,056 and 25,472; a large
// library product reaches 69). Tiles in 8 x 8 super-tiles per XCD share panels
// in L2.
// ---------------------------------------------------------------------------
constexpr int UT = 128, UK = 16, UP = 18;  // tile, columns per stage, LDS pitch
constexpr size_t kUpdateLds = (size_t)2 * 2 * UT * UP * 8;

__global__ void __launch_bounds__(512, 4) chol_update_kernel(MatBatch mb, int ld, int k0, int kw,
                                                             int base, int n, int nt, int tiles) {
    extern __shared__ __attribute__((aligned(16))) double sm[];
    const int t = (blockIdx.x & 7) * ((tiles + 7) >> 3) + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= ((tiles + 7) >> 3) || t >= tiles) return;
    int bj, bi;
    tri_super_tile(t, nt, bj, bi);  // bj <= bi
    double* __restrict__ A = mb.a[blockIdx.y];
    const int I0 = base + bi * UT, J0 = base + bj * UT;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wi = (wave & 1) * 64, wj = (wave >> 1) * 32;
    // the last tile row may reach past the matrix (n a multiple of 64): its rows
    // there are read as the last row and not written. The accumulators start
    // from minus the tile, so that its loads are in flight with the first stages
    doublex4 acc[4][2];
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                acc[m][q][v] = -A[(size_t)min(I0 + wi + 16 * m + (lane >> 4) + 4 * v, n - 1) * ld +
                                  min(J0 + wj + 16 * q + (lane & 15), n - 1)];
    // 128 rows x 8 pairs of columns a panel and stage, two pieces a thread
    const int r0 = tid >> 3, cc = 2 * (tid & 7);
    const double* pa[2];
    const double* pb[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        pa[u] = A + (size_t)min(I0 + r0 + 64 * u, n - 1) * ld + k0 + cc;
        pb[u] = A + (size_t)min(J0 + r0 + 64 * u, n - 1) * ld + k0 + cc;
    }
    doublex2 ra[2], rb[2];
    auto load = [&](int st) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            ra[u] = *reinterpret_cast<const doublex2*>(pa[u] + UK * st);
            rb[u] = *reinterpret_cast<const doublex2*>(pb[u] + UK * st);
        }
    };
    auto store = [&](int buf) {
        double* a = sm + buf * 2 * UT * UP;
        double* b = a + UT * UP;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            *reinterpret_cast<doublex2*>(a + (r0 + 64 * u) * UP + cc) = ra[u];
            *reinterpret_cast<doublex2*>(b + (r0 + 64 * u) * UP + cc) = rb[u];
        }
    };
    const int nst = kw / UK;
    load(0);
    store(0);
    load(min(1, nst - 1));
    __syncthreads();
    for (int st = 0; st < nst; ++st) {
        const double* a = sm + (st & 1) * 2 * UT * UP + (wi + (lane & 15)) * UP + (lane >> 4);
        const double* b = sm + (st & 1) * 2 * UT * UP + UT * UP + (wj + (lane & 15)) * UP + (lane >> 4);
        store((st + 1) & 1);
        load(min(st + 2, nst - 1));
#pragma unroll
        for (int ks = 0; ks < UK; ks += 4) {
            double x[4], y[2];
#pragma unroll
            for (int m = 0; m < 4; ++m) x[m] = a[16 * m * UP + ks];
#pragma unroll
            for (int q = 0; q < 2; ++q) y[q] = b[16 * q * UP + ks];
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int q = 0; q < 2; ++q)
                    acc[m][q] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[m], y[q], acc[m][q], 0, 0, 0);
        }
        __syncthreads();
    }
    const bool inside = bj < bi && I0 + UT <= n;
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int i = I0 + wi + 16 * m + (lane >> 4) + 4 * v;
                const int j = J0 + wj + 16 * q + (lane & 15);
                if (inside || (j <= i && i < n)) A[(size_t)i * ld + j] = -acc[m][q][v];
            }
}

// ---------------------------------------------------------------------------
// Triangular solves by 256-blocks with the inverses of the diagonal blocks:
// two launches a block (the block's own product, the update of the rest),
// each reading its part of the factor once. Vectors of the batch at stride n.
// (One-wave substitutions of 64-blocks, before, took 20 ms a solve at 13,056,
// these 2 ms for two systems, 10 us a launch; the read of the two factors takes
// 0.6 ms.) Loads carry no condition, so that a thread has 16 or 32 in flight.
// ---------------------------------------------------------------------------
// y_k = L_kk^{-1} z_k: y_r = sum_{c <= r} W[c][r] z_c, W the stored transposed
// inverse; 64 rows a workgroup, four column groups
__global__ void __launch_bounds__(256) fwd_diag_kernel(MatBatch mb, int ld, int n, int k0, int w,
                                                       const double* __restrict__ z,
                                                       double* __restrict__ y) {
    __shared__ double part[4][64];
    const double* __restrict__ L = mb.a[blockIdx.y];
    z += (size_t)n * blockIdx.y, y += (size_t)n * blockIdx.y;
    const int lane = threadIdx.x & 63, g = threadIdx.x >> 6;
    const int r = blockIdx.x * 64 + lane;
    double s = 0.0;
    // the groups interleave, so their work is even; loads without a condition,
    // 16 in flight (below the diagonal they read L and are dropped)
    for (int u0 = 0; u0 < 64 * blockIdx.x + 64; u0 += 64) {
        double v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) v[u] = L[(size_t)(k0 + u0 + 4 * u + g) * ld + k0 + r];
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const int c = u0 + 4 * u + g;
            s += c < r ? v[u] * z[k0 + c] : 0.0;
        }
    }
    part[g][lane] = s;
    __syncthreads();
    if (g == 0)
        y[k0 + r] = ((part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane])) +
                    z[k0 + r] / L[(size_t)(k0 + r) * ld + k0 + r];
}

// z_i -= sum_c L[i][k0 + c] y[k0 + c] below the block; a wave per four rows
__global__ void __launch_bounds__(256) fwd_update_kernel(MatBatch mb, int ld, int n, int k0, int w,
                                                         const double* __restrict__ y,
                                                         double* __restrict__ z) {
    const double* __restrict__ L = mb.a[blockIdx.y];
    z += (size_t)n * blockIdx.y, y += (size_t)n * blockIdx.y;
    const int lane = threadIdx.x & 63;
    const int i0 = k0 + w + (blockIdx.x * 4 + (threadIdx.x >> 6)) * 4;
    double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int c = 2 * lane + 128 * h;
        if (c >= w) continue;
        const doublex2 yv = *reinterpret_cast<const doublex2*>(y + k0 + c);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (i0 + q >= n) continue;
            const doublex2 l = *reinterpret_cast<const doublex2*>(L + (size_t)(i0 + q) * ld + k0 + c);
            s[q] += l.x * yv.x + l.y * yv.y;
        }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        for (int o = 32; o > 0; o >>= 1) s[q] += __shfl_xor(s[q], o);
        if (lane == 0 && i0 + q < n) z[i0 + q] -= s[q];
    }
}

// x_k = L_kk^{-T} y_k: x_c = sum_{r >= c} W[c][r] y_r; a wave per row of W
__global__ void __launch_bounds__(256) bwd_diag_kernel(MatBatch mb, int ld, int n, int k0, int w,
                                                       const double* __restrict__ y,
                                                       double* __restrict__ x) {
    const double* __restrict__ L = mb.a[blockIdx.y];
    x += (size_t)n * blockIdx.y, y += (size_t)n * blockIdx.y;
    const int lane = threadIdx.x & 63;
    const int c = blockIdx.x * 4 + (threadIdx.x >> 6);
    const double* row = L + (size_t)(k0 + c) * ld + k0;
    double s = 0.0;
#pragma unroll
    for (int h = 0; h < 4; ++h) {
        const int r = 64 * h + lane;
        if (r > c && r < w) s += row[r] * y[k0 + r];
    }
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (lane == 0) x[k0 + c] = s + y[k0 + c] / row[c];
}

// y_c -= sum_r L[k0 + r][c] x[k0 + r] left of the block; 64 columns a
// workgroup, four row groups
__global__ void __launch_bounds__(256) bwd_update_kernel(MatBatch mb, int ld, int n, int k0, int w,
                                                         const double* __restrict__ x,
                                                         double* __restrict__ y) {
    __shared__ double part[4][64];
    const double* __restrict__ L = mb.a[blockIdx.y];
    x += (size_t)n * blockIdx.y, y += (size_t)n * blockIdx.y;
    const int lane = threadIdx.x & 63, g = threadIdx.x >> 6;
    const int c = blockIdx.x * 64 + lane;
    double s = 0.0;
    if (64 * g < w)
#pragma unroll
        for (int u0 = 0; u0 < 64; u0 += 32) {
            double v[32];
#pragma unroll
            for (int u = 0; u < 32; ++u) v[u] = L[(size_t)(k0 + 64 * g + u0 + u) * ld + c];
#pragma unroll
            for (int u = 0; u < 32; ++u) s += v[u] * x[k0 + 64 * g + u0 + u];
        }
    part[g][lane] = s;
    __syncthreads();
    if (g == 0) y[c] -= (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]);
}

// r = b - (A + alpha I) x with the full symmetric A: one wave per row, lanes
// over the row (coalesced), FP64 with compensated (TwoSum) accumulation per
// lane and a compensated combination of the lane sums.
__device__ __forceinline__ void two_sum(double a, double b, double& s, double& e) {
    s = a + b;
    const double bb = s - a;
    e = (a - (s - bb)) + (b - bb);
}

__global__ void __launch_bounds__(256) residual_kernel(const double* __restrict__ A, int ld, int n,
                                                       MatBatch mb, const double* __restrict__ x,
                                                       const double* __restrict__ b, size_t b_stride,
                                                       double* __restrict__ r) {
    const double alpha = mb.alpha[blockIdx.y];
    x += (size_t)ld * blockIdx.y, r += (size_t)ld * blockIdx.y, b += b_stride * blockIdx.y;
    const int i = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (i >= n) return;
    const double* row = A + (size_t)i * ld;
    double s = 0.0, comp = 0.0;
    for (int c = lane; c < n; c += 64) {
        double t, e;
        two_sum(s, row[c] * x[c], t, e);
        s = t, comp += e;
    }
    for (int o = 32; o > 0; o >>= 1) {
        const double so = __shfl_xor(s, o), co = __shfl_xor(comp, o);
        double t, e;
        two_sum(s, so, t, e);
        s = t, comp += co + e;
    }
    if (lane == 0) r[i] = b[i] - ((s + comp) + alpha * x[i]);
}

// a copy of the lower triangle's 64-blocks of A with alpha on the first n
// diagonal elements
__global__ void __launch_bounds__(256) shifted_copy_kernel(const double* __restrict__ A, int ld,
                                                           int n, MatBatch mb) {
    double* __restrict__ out = mb.a[blockIdx.y];
    const int bi = blockIdx.x / (ld / SB), bj = blockIdx.x % (ld / SB);
    if (bj > bi) return;
    const double alpha = mb.alpha[blockIdx.y];
#pragma unroll 8
    for (int e = threadIdx.x; e < SB * SB / 2; e += 256) {
        const int r = bi * SB + (e >> 5), c = bj * SB + 2 * (e & 31);
        doublex2 v = *reinterpret_cast<const doublex2*>(A + (size_t)r * ld + c);
        if (r == c && r < n) v.x += alpha;
        if (r == c + 1 && r < n) v.y += alpha;
        *reinterpret_cast<doublex2*>(out + (size_t)r * ld + c) = v;
    }
}

__global__ void axpy_kernel(int n, int ld, const double* __restrict__ d, double* __restrict__ x) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const size_t k = (size_t)ld * blockIdx.y + i;
    if (i < n) x[k] += d[k];
}

// The n x n matrix src on an identity of order ld (rows of src are contiguous)
__global__ void __launch_bounds__(256) pad_system_kernel(const double* __restrict__ src, int n,
                                                         int ld, double* __restrict__ A) {
    const int i = blockIdx.x;
#pragma unroll 4
    for (int c = threadIdx.x; c < ld; c += 256)
        A[(size_t)i * ld + c] = i < n && c < n ? src[(size_t)i * n + c] : (i == c ? 1.0 : 0.0);
}

// The scaled normal equations straight from the accumulator's Gram of
// [X | y] (upper triangle valid, leading dimension ldg; column F holds X^T y):
// A[i][j] = G[i][j] / s[i] / s[j] (the reference's xtx /= s[:, None];
// xtx /= s[None, :]), zero for dropped columns, identity on the padding
// (i, j >= F), the full symmetric n_pad x n_pad matrix; b[i] = G[i][F] / s[i].
// 32 x 32 tiles; the lower tiles read the mirrored upper tile through LDS.
__global__ void __launch_bounds__(256) gram_system_kernel(const double* __restrict__ G, int ldg,
                                                          int F, const double* __restrict__ s,
                                                          const unsigned char* __restrict__ zero,
                                                          double* __restrict__ A, int lda,
                                                          double* __restrict__ b) {
    __shared__ double T[32][33];
    const int bi = blockIdx.y, bj = blockIdx.x;
    const int r0 = min(bi, bj) * 32, c0 = max(bi, bj) * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    for (int k = ty; k < 32; k += 8) {
        const int r = r0 + k, c = c0 + tx;
        T[k][tx] = (r < F && c < F) ? G[(size_t)r * ldg + c] : 0.0;
    }
    __syncthreads();
    for (int k = ty; k < 32; k += 8) {
        const int i = bi * 32 + k, j = bj * 32 + tx;
        double v;
        if (i >= F || j >= F) {
            v = i == j ? 1.0 : 0.0;
        } else if (zero[i] || zero[j]) {
            v = 0.0;
        } else {
            // element (min(i, j), max(i, j)) of the upper triangle
            const bool upper = bi < bj || (bi == bj && k <= tx);
            v = (upper ? T[k][tx] : T[tx][k]) / s[i] / s[j];
        }
        A[(size_t)i * lda + j] = v;
    }
    if (bj == 0 && threadIdx.x < 32) {
        const int i = bi * 32 + threadIdx.x;
        b[i] = (i < F && !zero[i]) ? G[(size_t)i * ldg + F] / s[i] : 0.0;
    }
}

// Rows [i0, i0 + rows) of the full symmetric F x F matrix, without the
// padding, from the accumulator's upper triangle, and X^T y from its column F:
// what a caller reads back is laid out here, so that one copy moves it. Mirrored
// on the host, the 2,264 columns' sums (41 MB) took 17.9 ms to read back; now
// 4.0 ms, which is the copy into the caller's fresh pages. 32 x 32 tiles as above. i0 is a multiple of 32.
__global__ void __launch_bounds__(256) gram_mirror_kernel(const double* __restrict__ G, int ldg,
                                                          int F, int i0, int rows,
                                                          double* __restrict__ out,
                                                          double* __restrict__ xty) {
    __shared__ double T[32][33];
    const int bi = blockIdx.y + i0 / 32, bj = blockIdx.x;
    const int r0 = min(bi, bj) * 32, c0 = max(bi, bj) * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    for (int k = ty; k < 32; k += 8) {
        const int r = r0 + k, c = c0 + tx;
        T[k][tx] = (r < F && c < F) ? G[(size_t)r * ldg + c] : 0.0;
    }
    __syncthreads();
    for (int k = ty; k < 32; k += 8) {
        const int i = bi * 32 + k, j = bj * 32 + tx;
        if (i >= i0 + rows || j >= F) continue;
        const bool upper = bi < bj || (bi == bj && k <= tx);
        out[(size_t)(i - i0) * F + j] = upper ? T[k][tx] : T[tx][k];
    }
    if (bj == 0 && threadIdx.x < 32) {
        const int i = bi * 32 + threadIdx.x;
        if (i < i0 + rows) xty[i] = G[(size_t)i * ldg + F];
    }
}

void launch_gram_mirror(hipStream_t st, const double* G, int ldg, int F, int i0, int rows,
                        double* out, double* xty) {
    const dim3 grid((F + 31) / 32, (rows + 31) / 32);
    gram_mirror_kernel<<<grid, 256, 0, st>>>(G, ldg, F, i0, rows, out, xty);
}

// y = A x for the full symmetric n x n system (one wave per row, lanes over
// the row: coalesced), FP64
__global__ void __launch_bounds__(256) symv_rows_kernel(const double* __restrict__ A, int lda,
                                                        int n, const double* __restrict__ x,
                                                        double* __restrict__ y) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= n) return;
    const double* a = A + (size_t)row * lda;
    double acc = 0.0;
    for (int c = lane; c < n; c += 64) acc += a[c] * x[c];
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
    if (lane == 0) y[row] = acc;
}

void launch_gram_system(hipStream_t st, const double* G, int ldg, int F, const double* s,
                        const unsigned char* zero, double* A, int lda, int n_pad, double* b) {
    const dim3 grid(n_pad / 32, n_pad / 32);
    gram_system_kernel<<<grid, 256, 0, st>>>(G, ldg, F, s, zero, A, lda, b);
}

void launch_symv(hipStream_t st, const double* A, int lda, int n, const double* x, double* y) {
    symv_rows_kernel<<<(n + 3) / 4, 256, 0, st>>>(A, lda, n, x, y);
}

// Right-looking over NB-wide panels, left-looking by 64 columns inside one.
// side: n_sys x n_pad x 64 values
void launch_cholesky(hipStream_t st, const MatBatch& mb, int n_sys, int ld, int n_pad,
                     double* side) {
    check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(&chol_step_kernel),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)kStepLds),
              "Cholesky shared memory");
    check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(&chol_update_kernel),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)kUpdateLds),
              "Cholesky shared memory");
    check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(&chol_inverse_kernel),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)kInvLds),
              "Cholesky shared memory");
    for (int k0 = 0; k0 < n_pad; k0 += NB) {
        const int kw = min(NB, n_pad - k0);
        for (int j0 = k0; j0 < k0 + kw; j0 += SB)
            chol_step_kernel<<<dim3((n_pad - j0) / SB, n_sys), 256, kStepLds, st>>>(mb, ld, k0, j0,
                                                                                         n_pad, side);
        const int base = k0 + kw;
        if (base >= n_pad) break;
        const int nt = (n_pad - base + UT - 1) / UT, tiles = nt * (nt + 1) / 2;
        chol_update_kernel<<<dim3((tiles + 7) / 8 * 8, n_sys), 512, kUpdateLds, st>>>(
            mb, ld, k0, kw, base, n_pad, nt, tiles);
    }
    chol_inverse_kernel<<<dim3((n_pad + NB - 1) / NB, n_sys), 256, kInvLds, st>>>(mb, ld, n_pad, side);
}

void launch_chol_solve(hipStream_t st, const MatBatch& mb, int n_sys, int ld, int n_pad, double* z,
                       double* y) {
    for (int k0 = 0; k0 < n_pad; k0 += NB) {
        const int w = min(NB, n_pad - k0), rest = n_pad - k0 - w;
        fwd_diag_kernel<<<dim3(w / 64, n_sys), 256, 0, st>>>(mb, ld, n_pad, k0, w, z, y);
        if (rest > 0)
            fwd_update_kernel<<<dim3((rest + 15) / 16, n_sys), 256, 0, st>>>(mb, ld, n_pad, k0, w, y, z);
    }
    for (int k0 = (n_pad - 1) / NB * NB; k0 >= 0; k0 -= NB) {
        const int w = min(NB, n_pad - k0);
        bwd_diag_kernel<<<dim3(w / 4, n_sys), 256, 0, st>>>(mb, ld, n_pad, k0, w, y, z);
        if (k0 > 0)
            bwd_update_kernel<<<dim3(k0 / 64, n_sys), 256, 0, st>>>(mb, ld, n_pad, k0, w, z, y);
    }
}

void launch_residual(hipStream_t st, const double* A, int ld, int n, const MatBatch& mb, int n_sys,
                     const double* x, const double* b, size_t b_stride, double* r) {
    residual_kernel<<<dim3((n + 3) / 4, n_sys), 256, 0, st>>>(A, ld, n, mb, x, b, b_stride, r);
}

void launch_shifted_copy(hipStream_t st, const double* A, int ld, int n, const MatBatch& mb,
                         int n_sys) {
    const int nb = ld / SB;
    shifted_copy_kernel<<<dim3(nb * nb, n_sys), 256, 0, st>>>(A, ld, n, mb);
}

void launch_pad_system(hipStream_t st, const double* src, int n, int n_pad, double* A) {
    pad_system_kernel<<<n_pad, 256, 0, st>>>(src, n, n_pad, A);
}

void launch_axpy(hipStream_t st, int n, int ld, int n_sys, const double* d, double* x) {
    axpy_kernel<<<dim3((n + 255) / 256, n_sys), 256, 0, st>>>(n, ld, d, x);
}

// padding granularity of the solve's matrices: whole 64-blocks
int solve_block() { return SB; }

}  // namespace plm
