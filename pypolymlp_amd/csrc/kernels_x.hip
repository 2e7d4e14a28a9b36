// HIP kernels of the X path for gfx950: the order parameters a_{nlm,tp}(i).
//
// Reference loop nest these kernels replace:
//   Local::compute_anlmtp_d (values, conjugate fill)  src/cxx/src/compute/local.cpp:116-217
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <stdexcept>
#include <type_traits>

#include "device_math.hpp"
#include "device_tables.hpp"
#include "kernels.hpp"
#include "pair_data.hpp"

namespace plm {

void check_hip(hipError_t e, const char* what);

// ---------------------------------------------------------------------------
// Order parameters a_{nlm,tp}(i) (noconj accumulation + conjugate fill).
// One workgroup per atom. skip_tol follows local.cpp:164 (f_n < 1e-20 skipped).
// ---------------------------------------------------------------------------
constexpr int kAnlmPairs = 16;

template <class T>
__global__ void __launch_bounds__(256) anlm_kernel(ModelDev md, BatchDev bd,
                                                   Cpx<T>* __restrict__ a_full, int a_stride,
                                                   int atom0, int n_atoms, int negate) {
    extern __shared__ unsigned char smem_raw[];
    const int ia = blockIdx.x;
    if (ia >= n_atoms) return;
    const int i = atom0 + ia;
    const int t1 = bd.types[i];
    const TypeDev& TT = md.t[t1];
    const PairLayout<T> L(md.n_fn, md.n_lmh, false);  // values only
    const int NPS = kAnlmPairs;  // pairs per chunk, one lane each
    T* pairs = reinterpret_cast<T*>(smem_raw);
    Cpx<T>* acc = reinterpret_cast<Cpx<T>*>(pairs + (size_t)NPS * L.stride);
    for (int h = threadIdx.x; h < TT.n_noconj; h += blockDim.x) acc[h] = {T(0), T(0)};
    const int p0 = bd.nb_off[i], p1 = bd.nb_off[i + 1];
    const int lmax = md.max_l;
    for (int c0 = p0; c0 < p1; c0 += NPS) {
        const int np = min(NPS, p1 - c0);
        __syncthreads();
        // X path: d = r_j - r_i + T (local.cpp:149); evaluation: the reversed
        // vector r_i - r_j - T (polymlp_eval.cpp:376-379)
        pairs_coop<T>(md, L, pairs, np, c0, bd, t1, 0, false, negate ? -1.0 : 1.0, lmax);
        for (int p = 0; p < np; ++p) {
            T* slot = pairs + (size_t)p * L.stride;
            const T* m = L.misc(slot);
            if (m[4] == T(0)) continue;
            const int tp = int(m[5]);
            const T* fn = L.fn(slot);
            const Cpx<T>* Y = L.Y(slot);
            const int h0 = TT.nc_tp_off[tp], h1 = TT.nc_tp_off[tp + 1];
            for (int h = h0 + threadIdx.x; h < h1; h += blockDim.x) {
                const T f = fn[TT.nc_tp_nid[h]];
                if (f < T(1e-20)) continue;
                const int key = TT.nc_tp_ylm[h];
                const int hd = TT.nc_tp_head[h];
                if (key < 0) {
                    acc[hd].re += f;
                } else {
                    acc[hd].re += f * Y[key].re;
                    acc[hd].im += f * Y[key].im;
                }
            }
        }
    }
    __syncthreads();
    Cpx<T>* out = a_full + (size_t)ia * a_stride;
    for (int k = threadIdx.x; k < TT.n_nlm; k += blockDim.x) {
        const Cpx<T> v = acc[TT.nlm_src[k]];
        if (TT.nlm_conj[k]) {
            const T cc = T(TT.nlm_sign[k]);
            out[k] = {cc * v.re, -cc * v.im};
        } else {
            out[k] = v;
        }
    }
}

// Order parameters with register sums (evaluation, at most NT Q heads per
// type, NT threads per atom): thread t owns the entries t + NT q (q < Q) of the
// atom type's list
// grouped by type pair, holds their type pair, radial index, Y key and head
// in registers for the whole atom, and adds f_n Y_lm of every pair of its
// entries' type pair into a register sum; the sums go to their heads at the
// end. Pairs are taken in the same order as anlm_kernel, so the sums are the
// same; the entry tables are read once per atom instead of once per pair and
// the LDS read-modify-write per pair and entry is gone.
template <class T, int Q, int NT>
__global__ void __launch_bounds__(NT) anlm_reg_kernel(ModelDev md, BatchDev bd,
                                                      Cpx<T>* __restrict__ a_full, int a_stride,
                                                      int atom0, int n_atoms, int negate) {
    extern __shared__ unsigned char smem_raw[];
    const int ia = blockIdx.x;
    if (ia >= n_atoms) return;
    const int i = atom0 + ia;
    const int t1 = bd.types[i];
    const TypeDev& TT = md.t[t1];
    const PairLayout<T> L(md.n_fn, md.n_lmh, false);  // values only
    const int NPS = kAnlmPairs;
    T* pairs = reinterpret_cast<T*>(smem_raw);
    Cpx<T>* acc = reinterpret_cast<Cpx<T>*>(pairs + (size_t)NPS * L.stride);
    const int tid = threadIdx.x;
    const int n_nc = TT.nc_tp_off[md.n_tp];
    int etp[Q], enid[Q], ekey[Q], ehd[Q];
    Cpx<T> a[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int h = tid + NT * q;
        etp[q] = -1, enid[q] = 0, ekey[q] = 0, ehd[q] = 0;
        a[q] = {T(0), T(0)};
        if (h < n_nc) {
            int tp = 0;
            while (TT.nc_tp_off[tp + 1] <= h) ++tp;
            etp[q] = tp, enid[q] = TT.nc_tp_nid[h], ekey[q] = TT.nc_tp_ylm[h];
            ehd[q] = TT.nc_tp_head[h];
        }
    }
    for (int h = tid; h < TT.n_noconj; h += blockDim.x) acc[h] = {T(0), T(0)};
    const int p0 = bd.nb_off[i], p1 = bd.nb_off[i + 1];
    const int lmax = md.max_l;
    for (int c0 = p0; c0 < p1; c0 += NPS) {
        const int np = min(NPS, p1 - c0);
        __syncthreads();
        // X path: d = r_j - r_i + T (local.cpp:149); evaluation: the reversed
        // vector r_i - r_j - T (polymlp_eval.cpp:376-379)
        pairs_coop<T>(md, L, pairs, np, c0, bd, t1, 0, false, negate ? -1.0 : 1.0, lmax);
        for (int p = 0; p < np; ++p) {
            T* slot = pairs + (size_t)p * L.stride;
            const T* m = L.misc(slot);
            if (m[4] == T(0)) continue;
            const int tp = int(m[5]);
            const T* fn = L.fn(slot);
            const Cpx<T>* Y = L.Y(slot);
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                if (etp[q] != tp) continue;
                const T f = fn[enid[q]];
                if (f < T(1e-20)) continue;
                if (ekey[q] < 0) {
                    a[q].re += f;
                } else {
                    const Cpx<T> y = Y[ekey[q]];
                    a[q].re += f * y.re;
                    a[q].im += f * y.im;
                }
            }
        }
    }
    __syncthreads();  // the zeroed heads, before the entries' sums land on theirs
#pragma unroll
    for (int q = 0; q < Q; ++q)
        if (etp[q] >= 0) acc[ehd[q]] = a[q];
    __syncthreads();
    Cpx<T>* out = a_full + (size_t)ia * a_stride;
    for (int k = threadIdx.x; k < TT.n_nlm; k += blockDim.x) {
        const Cpx<T> v = acc[TT.nlm_src[k]];
        if (TT.nlm_conj[k]) {
            const T cc = T(TT.nlm_sign[k]);
            out[k] = {cc * v.re, -cc * v.im};
        } else {
            out[k] = v;
        }
    }
}

// ---------------------------------------------------------------------------
// The same sums as a matrix product per atom, one workgroup of four waves:
//   a[(type, n)][key] = sum_p F[n][p] Y[key][p],
// F the radial functions (a row of another type's pairs masked to zero), Y the
// spherical harmonics, re and im in columns of their own, p the atom's
// neighbours, 64 at a time. A lane takes a pair; one or two waves take the
// columns m of Y (recurrences unrolled to LB, so their square roots are
// constants; the form above takes them, and a division each, per pair), the
// others the radial functions; both go to LDS as [row][pair] (pitch 66: the 16
// rows x 4 pairs of an MFMA operand are then on banks of their own), and 16 x 16
// x 4 MFMA tiles, dealt to the waves, Q at most each, add them up in registers.
// Bound by the functions of each pair (distance,
// angles, cos, exp: the matrix units take a fifth of the time), hence by waves
// in flight: four a SIMD (128 registers; with the 144 the compiler took 0.24 ms)
// and the angles and the cutoff function not in every wave (0.32 ms).
// Register sums -> this: 32,000 atoms of 50 neighbours, 165 heads 0.77 -> 0.20
// ms; 1,024 alloy atoms, 1,350 heads 0.17 -> 0.056 ms; 54 atoms 41 -> 7 us; 2,744
// atoms of 232 neighbours, pair model 0.15 -> 0.05 ms. FP64 only: an evaluation
// in FP32 (models past the LDS of the FP64 one) takes the forms above.
// ---------------------------------------------------------------------------
constexpr int kAnlmPitch = 66;
typedef double doublex4 __attribute__((ext_vector_type(4)));

// row of a lane's output element v of a 16 x 16 tile
__device__ __forceinline__ int anlm_row(int lane, int v) { return (lane >> 4) + 4 * v; }

template <int LB, int Q>
__global__ void __launch_bounds__(256, Q <= 4 ? 4 : 1) anlm_mfma_kernel(ModelDev md, BatchDev bd,
                                                        Cpx<double>* __restrict__ a_full,
                                                        int a_stride, int atom0, int negate) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    using T = double;
    using C = MathConst<T>;
    constexpr int P = kAnlmPitch;
    const int nfn = md.n_fn, ncol = 2 * max(1, md.n_lmh);
    T* F = reinterpret_cast<T*>(smem_raw);  // [n_fn][P]
    T* Y = F + (size_t)nfn * P;             // [ncol][P]
    __shared__ int group[64];
    const int ia = blockIdx.x;
    const int i = atom0 + ia;
    const int t1 = bd.types[i];
    const TypeDev& TT = md.t[t1];
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rt = (nfn + 15) / 16, ct = (ncol + 15) / 16;
    const int tiles = md.n_type * rt * ct;
    const int lmax = md.max_l;
    // waves on Y's columns, the others take the radial functions
    constexpr int NA = LB <= 4 ? 1 : 2;
    const int na = lmax < 0 ? 0 : NA;
    doublex4 acc[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) acc[q] = doublex4{0.0, 0.0, 0.0, 0.0};
    const int p0 = bd.nb_off[i], p1 = bd.nb_off[i + 1];
    for (int c0 = p0; c0 < p1; c0 += 64) {
        const int np = min(64, p1 - c0);
        if (c0 > p0) __syncthreads();  // the tiles have read the last chunk
        double dx = 0.0, dy = 0.0, dz = 0.0, dis = 0.0;
        int t2 = 0;
        if (lane < np) {
            const double* dk = bd.nb_d + 3 * (size_t)(c0 + lane);
            t2 = bd.types[bd.nb_j[c0 + lane]];
            // evaluation: the reversed vector r_i - r_j - T (polymlp_eval.cpp:376-379)
            const double sg = negate ? -1.0 : 1.0;
            dx = sg * dk[0], dy = sg * dk[1], dz = sg * dk[2];
            dis = sqrt(dx * dx + dy * dy + dz * dz);
        }
        const bool on = lane < np && dis < md.cutoff;
        if (w == 0) group[lane] = t2;
        if (w >= na) {
            const int tp = md.tp_of[t1 * md.n_type + t2];
            const int cnt = on ? md.rad_count[tp] : 0;
            const double* rp = md.rad + (size_t)tp * nfn * 2;
            const T fc = T(0.5) * (cospi(dis / md.cutoff) + T(1));
            for (int n = w - na; n < nfn; n += 4 - na) {
                const T beta = T(rp[2 * n]), x = T(dis) - T(rp[2 * n + 1]);
                const T f = dexp(-beta * x * x) * fc;
                F[n * P + lane] = n < cnt && !(f < T(1e-20)) ? f : T(0);
            }
            if (lmax < 0 && w < 2) Y[w * P + lane] = w == 0 ? T(1) : T(0);
        } else {
            const T x = T(dx), y = T(dy), z = T(dz), r = T(dis);
            const T ct_ = on ? z / r : T(1);
            T cp = T(1), sp = T(0);
            const T rho = sqrt(x * x + y * y);
            if (rho > T(0)) {
                const T inv = T(1) / rho;
                cp = x * inv, sp = y * inv;
            }
            const T st = dsqrt(T(1) - ct_ * ct_);
            T c = T(1), s = T(0);  // cos, sin (m phi) by the Chebyshev recurrence
            T c1 = T(1), c2 = cp, s1 = T(0), s2 = -sp, pmm = C::sqrt_inv_2pi;
            const T tc = T(2) * c2;
#pragma unroll
            for (int m = 0; m <= LB; ++m) {
                if (m > lmax) break;
                if (m >= 1) {
                    s = tc * s1 - s2;
                    c = tc * c1 - c2;
                    c2 = c1, c1 = c, s2 = s1, s1 = s;
                    pmm *= m == 1 ? -st * C::sqrt3div2
                                  : -dsqrt(T(1) + T(0.5) / T(m)) * st;
                }
                if (m % NA != w) continue;
                const T sign = (m % 2 == 1) ? T(-1) : T(1);
                T pa = T(0), pb = pmm;
#pragma unroll
                for (int l = m; l <= LB; ++l) {
                    if (l > lmax) break;
                    if (l == m + 1) {
                        const T pn = m == 0 ? ct_ * C::sqrt3 * C::sqrt_inv_2pi
                                            : dsqrt(T(2) * T(m) + T(3)) * ct_ * pb;
                        pa = pb, pb = pn;
                    } else if (l > m) {
                        const T ls = T(l * l), lm1s = T((l - 1) * (l - 1)), msq = T(m * m);
                        const T alm = dsqrt((T(4) * ls - T(1)) / (ls - msq));
                        const T blm = -dsqrt((lm1s - msq) / (T(4) * lm1s - T(1)));
                        const T pn = alm * (ct_ * pb + blm * pa);
                        pa = pb, pb = pn;
                    }
                    const int key = lm2i(l, -m) + l;
                    const T tmp = sign * pb * C::half_sqrt2;
                    Y[(2 * key) * P + lane] = on ? (m == 0 ? tmp : tmp * c) : T(0);
                    Y[(2 * key + 1) * P + lane] = on && m > 0 ? -tmp * s : T(0);
                }
            }
        }
        __syncthreads();
        const int rl = lane & 15, kl = lane >> 4;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int t = w + 4 * q;
            if (t >= tiles) break;
            const int g = t / (rt * ct), tr = t % (rt * ct) / ct, tcol = t % ct;
            // rows and columns past the end: any values, not read back
            const T* a = F + (size_t)min(16 * tr + rl, nfn - 1) * P + kl;
            const T* b = Y + (size_t)min(16 * tcol + rl, ncol - 1) * P + kl;
            for (int k = 0; k < np; k += 16) {
                T fa[4], fb[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int gu = group[k + 4 * u + kl];
                    fa[u] = a[k + 4 * u], fb[u] = b[k + 4 * u];
                    fa[u] = gu == g ? fa[u] : T(0);
                }
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    acc[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[u], fb[u], acc[q], 0, 0, 0);
            }
        }
    }
    __syncthreads();
    T* sums = F;  // [n_type][n_fn][ncol]
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int t = w + 4 * q;
        if (t >= tiles) break;
        const int g = t / (rt * ct), tr = t % (rt * ct) / ct, tcol = t % ct;
        const int col = 16 * tcol + (lane & 15);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int n = 16 * tr + anlm_row(lane, v);
            if (n < nfn && col < ncol) sums[((size_t)g * nfn + n) * ncol + col] = acc[q][v];
        }
    }
    __syncthreads();
    Cpx<T>* out = a_full + (size_t)ia * a_stride;
    for (int k = threadIdx.x; k < TT.n_nlm; k += 256) {
        const int at = TT.nlm_at[k];
        const T re = sums[at], im = sums[at + 1];
        const T cc = T(TT.nlm_sign[k]);
        out[k] = TT.nlm_conj[k] ? Cpx<T>{cc * re, -cc * im} : Cpx<T>{re, im};
    }
}

static size_t anlm_mfma_smem(const ModelDev& md) {
    const int ncol = 2 * std::max(1, md.n_lmh);
    return std::max((size_t)(md.n_fn + ncol) * kAnlmPitch, (size_t)md.n_type * md.n_fn * ncol) *
           sizeof(double);
}

static int anlm_mfma_tiles(const ModelDev& md) {
    return md.n_type * ((md.n_fn + 15) / 16) * ((2 * std::max(1, md.n_lmh) + 15) / 16);
}

// false: the model has Y columns past the unrolled ones, more tiles than four
// waves hold in registers (16 each) or rows past a CU's LDS, and the forms with
// sums per head below take it. Where it fits it is the faster one at every size
// tried (54 to 32,000 atoms, above).
static bool anlm_mfma_fits(const ModelDev& md) {
    return !getenv("PLM_ANLM_SHAPE") && md.max_l <= 12 && anlm_mfma_tiles(md) <= 4 * 16 &&
           anlm_mfma_smem(md) <= 156 * 1024;
}

static void launch_anlm_mfma(hipStream_t st, const ModelDev& md, const BatchDev& bd, void* a_full,
                      int a_stride, int atom0, int n_atoms, int negate) {
    const size_t sm = anlm_mfma_smem(md);
    auto go = [&](auto kernel) {
        check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)sm),
                  "anlm shared memory");
        kernel<<<n_atoms, 256, sm, st>>>(md, bd, reinterpret_cast<Cpx<double>*>(a_full), a_stride,
                                         atom0, negate);
    };
    const int q = (anlm_mfma_tiles(md) + 3) / 4;
    if (md.max_l <= 4 && q <= 4) go(&anlm_mfma_kernel<4, 4>);
    else if (md.max_l <= 8 && q <= 4) go(&anlm_mfma_kernel<8, 4>);
    else go(&anlm_mfma_kernel<12, 16>);
}

size_t anlm_smem(const ModelDev& md, int elem, int nthreads, int max_noconj) {
    const PairLayout<double> L(md.n_fn, md.n_lmh, false);
    return (size_t)nthreads * L.stride * elem + (size_t)max_noconj * 2 * elem;
}

bool anlm_fits(const ModelDev& md, bool fp64, int max_noconj) {
    return (fp64 && anlm_mfma_fits(md)) ||
           anlm_smem(md, fp64 ? 8 : 4, kAnlmPairs, max_noconj) <= 160 * 1024;
}

template <class T, int Q, int NT>
void launch_anlm_reg(hipStream_t st, const ModelDev& md, const BatchDev& bd, void* a_full,
                     int a_stride, int atom0, int n_atoms, size_t sm, int negate) {
    check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(&anlm_reg_kernel<T, Q, NT>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)sm),
              "anlm shared memory");
    anlm_reg_kernel<T, Q, NT><<<n_atoms, NT, sm, st>>>(md, bd, reinterpret_cast<Cpx<T>*>(a_full),
                                                       a_stride, atom0, n_atoms, negate);
}

// The product form above where the model fits it; else register sums with 2-4
// entries per thread (measured: 128 x 2 for 165 heads
// 0.96 ms per 32,000 atoms against 1.37 ms for 64 x 4 and 1.06 ms for 256 x 1;
// 512 x 3 for 1,350 heads 2.20 ms per 8,192 atoms against 2.73 ms for 256 x 8),
// up to 2,048 heads per type; LDS sums beyond
// PLM_ANLM_SHAPE=2x128|3x256|3x512|4x512|lds forces one form (an error where
// the type's heads do not fit it)
template <class T>
void launch_anlm_t(hipStream_t st, const ModelDev& md, const BatchDev& bd, void* a_full,
                   int a_stride, int atom0, int n_atoms, int max_noconj, int negate) {
    if (std::is_same<T, double>::value && anlm_mfma_fits(md)) {
        launch_anlm_mfma(st, md, bd, a_full, a_stride, atom0, n_atoms, negate);
        return;
    }
    const int B = 64;
    const size_t sm = anlm_smem(md, sizeof(T), kAnlmPairs, max_noconj);
    if (const char* e = getenv("PLM_ANLM_SHAPE")) {
        auto forced = [&](int cap) {
            if (max_noconj > cap)
                throw std::invalid_argument("PLM_ANLM_SHAPE: the model's heads exceed this form");
        };
        if (!strcmp(e, "2x128")) {
            forced(2 * 128);
            launch_anlm_reg<T, 2, 128>(st, md, bd, a_full, a_stride, atom0, n_atoms, sm, negate);
            return;
        } else if (!strcmp(e, "3x256")) {
            forced(3 * 256);
            launch_anlm_reg<T, 3, 256>(st, md, bd, a_full, a_stride, atom0, n_atoms, sm, negate);
            return;
        } else if (!strcmp(e, "3x512")) {
            forced(3 * 512);
            launch_anlm_reg<T, 3, 512>(st, md, bd, a_full, a_stride, atom0, n_atoms, sm, negate);
            return;
        } else if (!strcmp(e, "4x512")) {
            forced(4 * 512);
            launch_anlm_reg<T, 4, 512>(st, md, bd, a_full, a_stride, atom0, n_atoms, sm, negate);
            return;
        } else if (strcmp(e, "lds") != 0) {
            throw std::invalid_argument("PLM_ANLM_SHAPE: 2x128, 3x256, 3x512, 4x512 or lds");
        }
        // lds: the LDS sums below
    } else if (max_noconj <= 2 * 128) {
        launch_anlm_reg<T, 2, 128>(st, md, bd, a_full, a_stride, atom0, n_atoms, sm, negate);
        return;
    } else if (max_noconj <= 3 * 256) {
        launch_anlm_reg<T, 3, 256>(st, md, bd, a_full, a_stride, atom0, n_atoms, sm, negate);
        return;
    } else if (max_noconj <= 3 * 512) {
        launch_anlm_reg<T, 3, 512>(st, md, bd, a_full, a_stride, atom0, n_atoms, sm, negate);
        return;
    } else if (max_noconj <= 4 * 512) {
        launch_anlm_reg<T, 4, 512>(st, md, bd, a_full, a_stride, atom0, n_atoms, sm, negate);
        return;
    }
    check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(&anlm_kernel<T>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)sm),
              "anlm shared memory");
    anlm_kernel<T><<<n_atoms, B, sm, st>>>(md, bd, reinterpret_cast<Cpx<T>*>(a_full), a_stride,
                                           atom0, n_atoms, negate);
}

void launch_anlm(hipStream_t st, bool fp64, const ModelDev& md, const BatchDev& bd, void* a_full,
                 int a_stride, int atom0, int n_atoms, int max_noconj, int negate) {
    if (fp64) launch_anlm_t<double>(st, md, bd, a_full, a_stride, atom0, n_atoms, max_noconj, negate);
    else launch_anlm_t<float>(st, md, bd, a_full, a_stride, atom0, n_atoms, max_noconj, negate);
}

}  // namespace plm
