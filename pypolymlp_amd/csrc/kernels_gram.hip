// Gram accumulation C += X^T X (upper block triangle) on MFMA. The weighted
// targets sit in column F of X, so the same accumulation gives X^T y
// (C[:F, F]) and y^T y (C[F, F]) from exactly the X the Gram sees.
//
//   plain FP64 : v_mfma_f64_16x16x4_f64, FP64 accumulation (the reference's
//                numpy x.T @ x, src/pypolymlp/mlp_dev/core/utils_sequential.py:94-109).
//   mixed      : X in FP32, quantised per (row chunk of at most 4096 rows,
//                column) to a shared exponent E and three signed 7-bit
//                integer slices (the energy and stress rows in chunks of their
//                own, before the force rows),
//                x~ = 2^(E-7) (d0 + d1 2^-7 + d2 2^-14).
//                All nine slice products run on v_mfma_i32_32x32x32_i8 with
//                exact int32 accumulation, one accumulator per level s+t, and
//                are combined in FP64 once per chunk. The result is the exact
//                Gram of x~ (positive semidefinite, consistent with X^T y),
//                which the ill-conditioned ridge problem needs: a Gram that
//                drops products or rounds partial sums is indefinite at the
//                scale of the ridge parameter.
//
// X is row-major with leading dimension ld (>= F + 1, multiple of 128) and
// rows padded with zeros to a multiple of 64.
#include <hip/hip_runtime.h>

#include <stdexcept>

#include <algorithm>

#include "kernels.hpp"
#include "solve_batch.hpp"

namespace plm {

void check_hip(hipError_t e, const char* what);

typedef __attribute__((__vector_size__(4 * sizeof(double)))) double doublex4;
typedef double doublex2 __attribute__((ext_vector_type(2)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

// ---------------------------------------------------------------------------
// FP64: 128 x 128 output tile per 512-thread workgroup, each of the eight waves
// a 64 x 32 part (4 x 2 MFMA blocks, 64 accumulator registers), two workgroups
// a CU. 16 rows per stage through two LDS buffers (row pitch 144: the two rows
// that half an operand read spans fall into the two halves of the banks), the
// stage after next in registers. Bound by FP64 MFMA issue. A 64-wide tile reads
// its panels at 8 flops a byte, which held the kernel at 42 TFLOP/s; this one
// runs at 68 (F = 13,020, 35,190 rows: 139 -> 87 ms; a large library product
// reaches 69); consecutive tiles of an XCD share panels in its L2.
// Tiles tile0 .. tile0 + tiles; blockIdx.y: row split (launch_gram_f64), whose
// results go to part.
// ---------------------------------------------------------------------------
constexpr int G64_T = 128, G64_K = 16, G64_P = 144;
constexpr size_t kGram64Lds = (size_t)2 * 2 * G64_K * G64_P * 8;
constexpr int kGram64Slots = 512;  // workgroups resident at once (two a CU)

template <bool SPLIT>
__global__ void __launch_bounds__(512, 4) gram_f64_kernel(const double* __restrict__ X, int ld,
                                                          int rows, int rows_split, int nb,
                                                          int tile0, int tiles,
                                                          double* __restrict__ C, int ldc,
                                                          double* __restrict__ part) {
    extern __shared__ __attribute__((aligned(16))) double sm64[];
    const int per = (tiles + 7) >> 3;
    const int t = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per || t >= tiles) return;
    int bi, bj;
    tri_super_tile(tile0 + t, nb, bi, bj);
    const int I0 = bi * G64_T, J0 = bj * G64_T;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wi = (wave & 1) * 64, wj = (wave >> 1) * 32;
    doublex4 acc[4][2];
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int q = 0; q < 2; ++q) acc[m][q] = doublex4{0, 0, 0, 0};
    const int row0 = SPLIT ? blockIdx.y * rows_split : 0;
    const int nst = (SPLIT ? min(rows_split, rows - row0) : rows) / G64_K;
    // 16 rows x 64 pairs of columns a panel and stage, two pieces a thread
    const double* pa = X + (size_t)(row0 + wave) * ld + I0 + 2 * lane;
    const double* pb = X + (size_t)(row0 + wave) * ld + J0 + 2 * lane;
    doublex2 ra[2], rb[2];
    auto load = [&](int st) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            ra[u] = *reinterpret_cast<const doublex2*>(pa + (size_t)(G64_K * st + 8 * u) * ld);
            rb[u] = *reinterpret_cast<const doublex2*>(pb + (size_t)(G64_K * st + 8 * u) * ld);
        }
    };
    auto store = [&](int buf) {
        double* a = sm64 + buf * 2 * G64_K * G64_P + wave * G64_P + 2 * lane;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            *reinterpret_cast<doublex2*>(a + 8 * u * G64_P) = ra[u];
            *reinterpret_cast<doublex2*>(a + (G64_K + 8 * u) * G64_P) = rb[u];
        }
    };
    load(0);
    store(0);
    load(min(1, nst - 1));
    __syncthreads();
    for (int st = 0; st < nst; ++st) {
        const double* a = sm64 + (st & 1) * 2 * G64_K * G64_P + (lane >> 4) * G64_P + wi + (lane & 15);
        const double* b = a + G64_K * G64_P - wi + wj;
        store((st + 1) & 1);
        load(min(st + 2, nst - 1));
#pragma unroll
        for (int ks = 0; ks < G64_K; ks += 4) {
            double x[4], y[2];
#pragma unroll
            for (int m = 0; m < 4; ++m) x[m] = a[ks * G64_P + 16 * m];
#pragma unroll
            for (int q = 0; q < 2; ++q) y[q] = b[ks * G64_P + 16 * q];
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int q = 0; q < 2; ++q)
                    acc[m][q] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[m], y[q], acc[m][q], 0, 0, 0);
        }
        __syncthreads();
    }
    // D[l/16 + 4v][l%16] of each 16 x 16 block
    const int i0 = wi + (lane >> 4), j0 = wj + (lane & 15);
    if constexpr (SPLIT) {
        double* o = part + ((size_t)blockIdx.y * tiles + t) * G64_T * G64_T + i0 * G64_T + j0;
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int v = 0; v < 4; ++v) o[(16 * m + 4 * v) * G64_T + 16 * q] = acc[m][q][v];
    } else {
        double* o = C + (size_t)(I0 + i0) * ldc + J0 + j0;
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            double c[2][4];
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int v = 0; v < 4; ++v) c[q][v] = o[(size_t)(16 * m + 4 * v) * ldc + 16 * q];
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    o[(size_t)(16 * m + 4 * v) * ldc + 16 * q] = c[q][v] + acc[m][q][v];
        }
    }
}

// C += the splits' tiles, in their order
__global__ void __launch_bounds__(256) gram_f64_sum_kernel(const double* __restrict__ part, int nb,
                                                           int tile0, int tiles, int splits,
                                                           double* __restrict__ C, int ldc) {
    const int t = blockIdx.x;
    int bi, bj;
    tri_super_tile(tile0 + t, nb, bi, bj);
    const int e = blockIdx.y * 512 + 2 * threadIdx.x;  // two of the tile's elements
    doublex2 s = {0.0, 0.0};
#pragma unroll 4
    for (int k = 0; k < splits; ++k)
        s += *reinterpret_cast<const doublex2*>(part + ((size_t)k * tiles + t) * G64_T * G64_T + e);
    doublex2* c = reinterpret_cast<doublex2*>(C + (size_t)(bi * G64_T + e / G64_T) * ldc +
                                              bj * G64_T + e % G64_T);
    *c += s;
}

// ---------------------------------------------------------------------------
// Mixed: quantisation
// ---------------------------------------------------------------------------
constexpr int kQChunk = 4096;  // rows sharing one exponent per column (at most)
constexpr int kQK = 32;        // rows per K step (one i8 MFMA)

// Row q of the quantised matrix is row rmap[q] of X (a zero row where
// rmap[q] < 0). The energy and stress rows of a sub-batch come first, then the
// force rows: an energy row sums a feature over all N atoms of its structure,
// so a chunk shared with force rows would set their exponent about N times too
// high. The Gram does not depend on the row order. Chunk 0 holds the first h0
// rows (a multiple of 64, at most kQChunk), chunk k > 0 the kQChunk rows from
// h0 + (k - 1) kQChunk, so the energy and stress rows end on a chunk boundary.
__host__ __device__ __forceinline__ int chunk_of(int q, int h0) {
    return q < h0 ? 0 : 1 + (q - h0) / kQChunk;
}
__host__ __device__ __forceinline__ int n_chunks_of(int rows, int h0) {
    return rows <= h0 ? 1 : 1 + (rows - h0 + kQChunk - 1) / kQChunk;
}
template <class T>
__device__ __forceinline__ T xrow(const T* __restrict__ X, const int* __restrict__ rmap, int q,
                                  int ld, int c) {
    const int r = rmap[q];
    return r >= 0 ? X[(size_t)r * ld + c] : T(0);
}
__device__ __forceinline__ int exponent_of(float m) {
    int e = 0;
    if (m > 0.f) (void)frexpf(m, &e);
    return e;
}
__device__ __forceinline__ int exponent_of(double m) {
    int e = 0;
    if (m > 0.0) (void)frexp(m, &e);
    return e;
}

// E[chunk][c]: smallest E with |x| < 2^E over the chunk's rows (0 for a zero column).
// 64 columns per workgroup, four row phases of 64 threads; each thread reads
// the row indices of its next eight rows, then keeps their eight loads in
// flight (the maximum is order independent, so the result does not depend on
// the split)
template <class T>
__global__ void __launch_bounds__(256) colexp_kernel(const T* __restrict__ X,
                                                     const int* __restrict__ rmap, int ld, int rows,
                                                     int h0, int ncols, int* __restrict__ E) {
    __shared__ T part[4][64];
    const int cx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    const int c = blockIdx.x * 64 + cx;
    const int chunk = blockIdx.y;
    const int r0 = chunk == 0 ? 0 : h0 + (chunk - 1) * kQChunk;
    const int r1 = min(rows, chunk == 0 ? h0 : r0 + kQChunk);
    T m[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) m[u] = T(0);
    if (c < ncols) {
        int r = r0 + ty;
        // the next batch's row indices load while this batch's rows of X do
        int rn[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) rn[u] = r + 28 < r1 ? rmap[r + 4 * u] : -1;
        for (; r + 28 < r1; r += 32) {
            int rr[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) rr[u] = rn[u];
            if (r + 60 < r1) {
#pragma unroll
                for (int u = 0; u < 8; ++u) rn[u] = rmap[r + 32 + 4 * u];
            }
            T v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = rr[u] >= 0 ? X[(size_t)rr[u] * ld + c] : T(0);
#pragma unroll
            for (int u = 0; u < 8; ++u) m[u] = fmax(m[u], fabs(v[u]));
        }
        for (; r < r1; r += 4) m[0] = fmax(m[0], fabs(xrow(X, rmap, r, ld, c)));
    }
#pragma unroll
    for (int u = 1; u < 8; ++u) m[0] = fmax(m[0], m[u]);
    part[ty][cx] = m[0];
    __syncthreads();
    if (ty == 0 && c < ncols) {
        const T m = fmax(fmax(part[0][cx], part[1][cx]), fmax(part[2][cx], part[3][cx]));
        E[(size_t)chunk * ld + c] = exponent_of(m);
    }
}

// Q[s][rb][c][k] (int8): slice s of x[rmap[32 rb + k]][c], k-contiguous per
// column so that 16 bytes are one lane's MFMA operand.
template <class T>
__global__ void quantize_kernel(const T* __restrict__ X, const int* __restrict__ rmap, int ld,
                                int rows_pad, int h0, int ncols, const int* __restrict__ E,
                                signed char* __restrict__ Q) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    const int rb = blockIdx.y;
    if (c >= ncols) return;
    const int nrb = rows_pad / kQK;
    const int e = E[(size_t)chunk_of(rb * kQK, h0) * ld + c];
    const size_t plane = (size_t)nrb * ld * kQK;
    signed char* q = Q + ((size_t)rb * ld + c) * kQK;
    // the block's 32 row indices (uniform) first, then all 32 loads of X in flight
    int rr[kQK];
#pragma unroll
    for (int k = 0; k < kQK; ++k) rr[k] = rmap[rb * kQK + k];
    T xv[kQK];
#pragma unroll
    for (int k = 0; k < kQK; ++k) xv[k] = rr[k] >= 0 ? X[(size_t)rr[k] * ld + c] : T(0);
#pragma unroll
    for (int k0 = 0; k0 < kQK; k0 += 16) {
        union {
            signed char b[16];
            v4i v;
        } d0, d1, d2;
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            const T x = xv[k0 + k];
            const T m = ldexp(x, 7 - e);  // |m| < 128
            const T t0 = trunc(m);
            const T r1 = (m - t0) * T(128);  // exact
            const T t1 = trunc(r1);
            const T r2 = (r1 - t1) * T(128);  // exact
            const T t2 = fmin(fmax(rint(r2), T(-127)), T(127));
            d0.b[k] = (signed char)t0, d1.b[k] = (signed char)t1, d2.b[k] = (signed char)t2;
        }
        *reinterpret_cast<v4i*>(q + k0) = d0.v;
        *reinterpret_cast<v4i*>(q + plane + k0) = d1.v;
        *reinterpret_cast<v4i*>(q + 2 * plane + k0) = d2.v;
    }
}

// ---------------------------------------------------------------------------
// Mixed: 128 (i) x 64 (j) output tile per 512-thread workgroup; each of the 8
// waves owns one 32x32 block with five int32 accumulators (levels s + t =
// 0..4), so two waves run per SIMD. Stages of 64 rows through two LDS buffers
// (48-byte column stride, b128 reads without bank conflicts). In each stage a
// wave reads its operands, stores the next stage (loaded into registers one
// stage earlier) into the other buffer and issues the loads of the stage after;
// the LDS and global instructions are interleaved with the 18 MFMAs. Per
// 4096-row chunk the int32 levels are combined into FP64 sums held in
// registers; C is read and written once, at the end.
// ---------------------------------------------------------------------------
constexpr int GI_TI = 128;
constexpr int GI_TJ = 64;
constexpr int GI_NT = 512;                       // threads per workgroup
constexpr int GI_CS = 48;                        // LDS bytes per column and 32-row block
constexpr int GI_RB = 2;                         // 32-row blocks per stage
constexpr int GI_A = 3 * GI_RB * GI_TI * GI_CS;  // A panel bytes per stage
constexpr int GI_B = 3 * GI_RB * GI_TJ * GI_CS;  // B panel bytes per stage
constexpr int GI_PA = 3 * GI_RB * GI_TI * 2;     // 16-byte A pieces per stage
constexpr int GI_PB = 3 * GI_RB * GI_TJ * 2;     // 16-byte B pieces per stage
constexpr int GI_LA = (GI_PA + GI_NT - 1) / GI_NT;  // A pieces per thread
constexpr int GI_LB = (GI_PB + GI_NT - 1) / GI_NT;  // B pieces per thread
constexpr int GI_MFMA = 9 * GI_RB;               // MFMAs per wave and stage
static_assert(GI_PA % 64 == 0 && GI_PB % 64 == 0 && GI_TJ % 32 == 0,
              "staging pieces come in runs of 64 (32 columns x 2 halves)");

// Tile order: workgroups are dealt to the 8 XCDs round robin; each XCD runs
// one super-tile of 4 x 8 tiles (512 x 512 outputs) at a time, so the panels
// of concurrently running tiles are shared in its L2. Super-tiles (SI, SJ),
// SJ >= SI, cover the upper triangle; tiles below it return at once.
__device__ __forceinline__ bool tile_index_i8(int b, int nbi, int& bi, int& bj) {
    const int xcd = b & 7, k = b >> 3;
    const int sup = (k >> 5) * 8 + xcd, loc = k & 31;
    const int nsi = (nbi + 3) / 4;
    int r = 0, rem = sup;
    while (r < nsi && rem >= nsi - r) rem -= nsi - r, ++r;
    if (r >= nsi) return false;
    bi = r * 4 + (loc >> 3);
    bj = (r + rem) * 8 + (loc & 7);
    return bi < nbi && bj < 2 * nbi && bj >= 2 * bi;
}

static long gram_i8_grid(int nbi) {
    const long nsi = (nbi + 3) / 4, nsup = nsi * (nsi + 1) / 2;
    return (nsup + 7) / 8 * 8 * 32;
}

size_t gram_i8_smem() { return 2 * (size_t)(GI_A + GI_B); }

__global__ void __launch_bounds__(GI_NT) gram_i8_kernel(const signed char* __restrict__ Q, int ld,
                                                        int rows_pad, int h0, int nbi,
                                                        const int* __restrict__ E,
                                                        double* __restrict__ C, int ldc) {
    extern __shared__ __attribute__((aligned(16))) signed char smem_i8[];
    int bi, bj;
    if (!tile_index_i8(blockIdx.x, nbi, bi, bj)) return;
    const int I0 = bi * GI_TI, J0 = bj * GI_TJ;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wi = (wave & 3) * 32, wj = (wave >> 2) * 32;
    const int nrb = rows_pad / kQK;
    const int nst = nrb / GI_RB;
    const size_t plane = (size_t)nrb * ld * kQK;
    v16i acc[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) acc[k] = v16i{};
    double sacc[16];
#pragma unroll
    for (int v = 0; v < 16; ++v) sacc[v] = 0.0;
    // piece p -> ((s * GI_RB + rbo) * cols + col) * 2 + half
    // within each run of 64 pieces, pieces 0-31 are the first 16-byte halves of
    // 32 consecutive columns and pieces 32-63 their second halves, so the 16
    // lanes of one LDS store pass write 16 columns of one half (distinct banks
    // at the 48-byte column stride, as the operand reads)
    auto piece = [&](int p, int cols, int& half, int& col, int& sr) {
        const int q = (p >> 6) * 32 + (p & 31);
        half = (p >> 5) & 1, col = q % cols, sr = q / cols;
    };
    auto g_off = [&](int p, int cols, int col0, int st) -> size_t {
        int half, col, sr;
        piece(p, cols, half, col, sr);
        const int s = sr / GI_RB, rbo = sr % GI_RB;
        return s * plane + ((size_t)(st * GI_RB + rbo) * ld + col0 + col) * kQK + 16 * half;
    };
    auto l_off = [&](int p, int cols) -> int {
        int half, col, sr;
        piece(p, cols, half, col, sr);
        return (sr * cols + col) * GI_CS + 16 * half;
    };
    // thread pieces past a panel's end wrap around (branch-free): such a
    // thread loads and stores a copy of a piece another thread stores, the
    // same value into the same slot
    v4i ra[GI_LA], rb[GI_LB];
    auto load = [&](int st) {
#pragma unroll
        for (int r = 0; r < GI_LA; ++r)
            ra[r] = *reinterpret_cast<const v4i*>(Q + g_off((tid + GI_NT * r) % GI_PA, GI_TI, I0, st));
#pragma unroll
        for (int r = 0; r < GI_LB; ++r)
            rb[r] = *reinterpret_cast<const v4i*>(Q + g_off((tid + GI_NT * r) % GI_PB, GI_TJ, J0, st));
    };
    auto store = [&](int buf) {
        signed char* A = smem_i8 + (size_t)buf * (GI_A + GI_B);
        signed char* B = A + GI_A;
#pragma unroll
        for (int r = 0; r < GI_LA; ++r)
            *reinterpret_cast<v4i*>(A + l_off((tid + GI_NT * r) % GI_PA, GI_TI)) = ra[r];
#pragma unroll
        for (int r = 0; r < GI_LB; ++r)
            *reinterpret_cast<v4i*>(B + l_off((tid + GI_NT * r) % GI_PB, GI_TJ)) = rb[r];
    };
    // x~_i x~_j = 2^(E_i + E_j - 14) sum_k acc_k 2^(-7k): exact int32 sums
    // combined in FP64; D[(v%4) + 8(v/4) + 4(l/32)][l%32]
    const int i0 = I0 + wi + 4 * (lane >> 5);
    const int j = J0 + wj + (lane & 31);
    auto flush = [&](int chunk) {
        const int* Ec = E + (size_t)chunk * ld;
        const int ej = Ec[j];
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int di = (v & 3) + 8 * (v >> 2);
            double t = double(acc[4][v]);
            t = t * 0.0078125 + double(acc[3][v]);
            t = t * 0.0078125 + double(acc[2][v]);
            t = t * 0.0078125 + double(acc[1][v]);
            t = t * 0.0078125 + double(acc[0][v]);
            sacc[v] += ldexp(t, Ec[i0 + di] + ej - 14);
        }
#pragma unroll
        for (int k = 0; k < 5; ++k) acc[k] = v16i{};
    };
    const int st_per_chunk = kQChunk / (kQK * GI_RB);
    const int h0s = h0 / (kQK * GI_RB);  // stages of chunk 0
    const int nchunk = nst <= h0s ? 1 : 1 + (nst - h0s + st_per_chunk - 1) / st_per_chunk;
    load(0);
    store(0);
    load(nst > 1 ? 1 : 0);
    __syncthreads();
    for (int ch = 0; ch < nchunk; ++ch) {
        const int s1 = min(nst, h0s + ch * st_per_chunk);
        for (int st = ch == 0 ? 0 : h0s + (ch - 1) * st_per_chunk; st < s1; ++st) {
            const signed char* A = smem_i8 + (size_t)(st & 1) * (GI_A + GI_B);
            const signed char* B = A + GI_A;
            // lane -> column (lane % 32) of its block, k half (lane / 32)
            v4i a[GI_RB][3], b[GI_RB][3];
#pragma unroll
            for (int rbo = 0; rbo < GI_RB; ++rbo)
#pragma unroll
                for (int s = 0; s < 3; ++s) {
                    a[rbo][s] = *reinterpret_cast<const v4i*>(
                        A + ((s * GI_RB + rbo) * GI_TI + wi + (lane & 31)) * GI_CS + 16 * (lane >> 5));
                    b[rbo][s] = *reinterpret_cast<const v4i*>(
                        B + ((s * GI_RB + rbo) * GI_TJ + wj + (lane & 31)) * GI_CS + 16 * (lane >> 5));
                }
            // stage st + 1 into the other buffer (last read in iteration st - 1),
            // then the loads of stage st + 2 (past the end: the last stage again)
            store((st + 1) & 1);
            load(min(st + 2, nst - 1));
            // issue order: the k-th product of every level before any (k+1)-th
            constexpr int kS[3][5] = {{0, 0, 0, 1, 2}, {-1, 1, 1, 2, -1}, {-1, -1, 2, -1, -1}};
#pragma unroll
            for (int rbo = 0; rbo < GI_RB; ++rbo)
#pragma unroll
                for (int k = 0; k < 3; ++k)
#pragma unroll
                    for (int lvl = 0; lvl < 5; ++lvl) {
                        const int s = kS[k][lvl];
                        if (s < 0) continue;
                        acc[lvl] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[rbo][s], b[rbo][lvl - s],
                                                                         acc[lvl], 0, 0, 0);
                    }
            // schedule: the first row block's operands, then one MFMA per LDS
            // read of the second row block, per LDS store, per global load
            __builtin_amdgcn_sched_group_barrier(0x100, 3 * 2, 0);
#pragma unroll
            for (int i = 0; i < 3 * 2; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
#pragma unroll
            for (int i = 0; i < GI_LA + GI_LB; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
            }
#pragma unroll
            for (int i = 0; i < GI_LA + GI_LB; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x008, GI_MFMA - 6 - 2 * (GI_LA + GI_LB), 0);
            __syncthreads();
        }
        flush(ch);
    }
    double* cb = C + (size_t)i0 * ldc + j;
#pragma unroll
    for (int v = 0; v < 16; ++v) cb[(size_t)((v & 3) + 8 * (v >> 2)) * ldc] += sacc[v];
}

// y (FP64, one value per row) into column col of X (FP32 or FP64)
template <class T>
__global__ void set_column_kernel(T* __restrict__ X, int ld, int col, const double* __restrict__ y,
                                  int rows) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r < rows) X[(size_t)r * ld + col] = T(y[r]);
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
void launch_set_column(hipStream_t st, bool fp64, void* X, int ld, int col, const double* y,
                       int rows) {
    const int B = 256;
    if (fp64)
        set_column_kernel<double><<<(rows + B - 1) / B, B, 0, st>>>(reinterpret_cast<double*>(X),
                                                                    ld, col, y, rows);
    else
        set_column_kernel<float><<<(rows + B - 1) / B, B, 0, st>>>(reinterpret_cast<float*>(X), ld,
                                                                   col, y, rows);
}

size_t gram_quant_bytes(int rows_pad, int h0, int ld) {
    return 3 * (size_t)rows_pad * ld + (size_t)n_chunks_of(rows_pad, h0) * ld * sizeof(int);
}

// The FP64 Gram's tiles go in whole rounds of resident workgroups; the rows of
// the remaining tiles are split so that their round, too, fills the chip (F =
// 13,020: 5,253 tiles are 10 rounds and 133 tiles, and an eleventh round cost
// 1 of 88 ms; F = 2,277: 171 tiles in one launch left 85 CUs idle, 5.9 ms for
// 33,800 rows against 3.5 ms in 11 splits). Each split keeps at least 512 rows.
static int gram_f64_splits(int tiles, int rows) {
    const int per = (tiles + 7) / 8, slots = kGram64Slots / 8;  // of one XCD
    int best = 1;
    double cost = 1e30;
    for (int s = 1; s <= 32 && (s == 1 || rows / s >= 512); ++s) {
        // rounds of 1 / s of the rows each, and the traffic of the partial tiles
        const double c = (double)((per * s + slots - 1) / slots) / s + 0.002 * s;
        if (c < cost) cost = c, best = s;
    }
    return best;
}

size_t gram_f64_part_bytes(int rows_pad, int F_pad) {
    const int nb = F_pad / G64_T, rest = nb * (nb + 1) / 2 % kGram64Slots;
    const int splits = gram_f64_splits(rest, rows_pad);
    return splits == 1 ? 0 : (size_t)splits * rest * G64_T * G64_T * 8;
}

void launch_gram_f64(hipStream_t st, const double* X, int ld, int rows_pad, int F_pad, double* C,
                     int ldc, void* part) {
    if (F_pad % G64_T || rows_pad % G64_K) throw std::invalid_argument("FP64 Gram tile sizes");
    const int nb = F_pad / G64_T, tiles = nb * (nb + 1) / 2;
    check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(&gram_f64_kernel<false>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)kGram64Lds),
              "Gram shared memory");
    check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(&gram_f64_kernel<true>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)kGram64Lds),
              "Gram shared memory");
    const int rest = tiles % kGram64Slots;
    int splits = rest > 0 ? gram_f64_splits(rest, rows_pad) : 1;
    const int whole = splits == 1 ? tiles : tiles - rest;
    if (whole > 0)
        gram_f64_kernel<false><<<(whole + 7) / 8 * 8, 512, kGram64Lds, st>>>(
            X, ld, rows_pad, rows_pad, nb, 0, whole, C, ldc, nullptr);
    if (splits == 1) return;
    const int rs = ((rows_pad + splits - 1) / splits + G64_K - 1) / G64_K * G64_K;
    splits = (rows_pad + rs - 1) / rs;  // none is empty
    double* p = static_cast<double*>(part);
    gram_f64_kernel<true><<<dim3((rest + 7) / 8 * 8, splits), 512, kGram64Lds, st>>>(
        X, ld, rows_pad, rs, nb, whole, rest, C, ldc, p);
    gram_f64_sum_kernel<<<dim3(rest, G64_T * G64_T / 512), 256, 0, st>>>(p, nb, whole, rest, splits,
                                                                         C, ldc);
}

int gram_chunk_rows() { return kQChunk; }

void launch_gram_quantize(hipStream_t st, bool x_fp64, const void* X, const int* rmap, int ld,
                          int rows_pad, int h0, int F_pad, void* quant) {
    if (h0 < kQK * GI_RB || h0 > kQChunk || h0 % (kQK * GI_RB) || rows_pad % (kQK * GI_RB))
        throw std::invalid_argument("quantisation chunk rows");
    const int n_chunks = n_chunks_of(rows_pad, h0);
    signed char* Q = reinterpret_cast<signed char*>(quant);
    int* E = reinterpret_cast<int*>(Q + 3 * (size_t)rows_pad * ld);
    const int B = 256;
    const dim3 ge((F_pad + 63) / 64, n_chunks), gq((F_pad + B - 1) / B, rows_pad / kQK);
    if (x_fp64) {
        const double* Xd = static_cast<const double*>(X);
        colexp_kernel<double><<<ge, 256, 0, st>>>(Xd, rmap, ld, rows_pad, h0, F_pad, E);
        quantize_kernel<double><<<gq, B, 0, st>>>(Xd, rmap, ld, rows_pad, h0, F_pad, E, Q);
    } else {
        const float* Xf = static_cast<const float*>(X);
        colexp_kernel<float><<<ge, 256, 0, st>>>(Xf, rmap, ld, rows_pad, h0, F_pad, E);
        quantize_kernel<float><<<gq, B, 0, st>>>(Xf, rmap, ld, rows_pad, h0, F_pad, E, Q);
    }
}

void launch_gram_i8(hipStream_t st, int ld, int rows_pad, int h0, int F_pad, const void* quant,
                    double* C, int ldc) {
    const signed char* Q = reinterpret_cast<const signed char*>(quant);
    const int* E = reinterpret_cast<const int*>(Q + 3 * (size_t)rows_pad * ld);
    const int nbi = F_pad / GI_TI;
    const size_t sm = gram_i8_smem();
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&gram_i8_kernel),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)sm);
    gram_i8_kernel<<<gram_i8_grid(nbi), GI_NT, sm, st>>>(Q, ld, rows_pad, h0, nbi, E, C, ldc);
}

}  // namespace plm
