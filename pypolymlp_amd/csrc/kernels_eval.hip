// HIP kernels of PolymlpEval (energy, forces, stress) for gfx950.
//
// Reference loop nests:
//   PolymlpEval::compute_sum_of_prod_anlmtp   src/cxx/src/compute/polymlp_eval.cpp:337-404
//   Potential::compute_sum_of_prod_anlmtp     src/cxx/src/polymlp/polymlp_potential.cpp:235-321
//                                             (here as a gradient by features, then by heads)
//   PolymlpEval::eval_gtinv (half-pair loop)  polymlp_eval.cpp:182-291
//   PolymlpEval::eval_pair / compute_sum_of_prod_antp  polymlp_eval.cpp:46-180,
//                                             polymlp_potential.cpp:203-233
//   collect_properties                        polymlp_eval.cpp:293-335
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <stdexcept>

#include "device_math.hpp"
#include "device_tables.hpp"
#include "eval_tables.hpp"
#include "kernels.hpp"
#include "pair_data.hpp"

namespace plm {

void check_hip(hipError_t e, const char* what);

template <class T> struct EvalTab;  // the tables' coefficients by precision
template <> struct EvalTab<double> {
    __device__ static const double* value(const EvalTypeDev& e) { return e.vq_c; }
    __device__ static const double2* poly(const EvalTypeDev& e) { return e.pf_c; }
    __device__ static const double* term(const EvalTypeDev& e) { return e.tq_c; }
};
template <> struct EvalTab<float> {
    __device__ static const float* value(const EvalTypeDev& e) { return e.vq_cf; }
    __device__ static const float2* poly(const EvalTypeDev& e) { return e.pf_cf; }
    __device__ static const float* term(const EvalTypeDev& e) { return e.tq_cf; }
};

// product of the order parameters of a value term (16-bit keys, absent ones
// point at the constant 1)
template <class T>
__device__ __forceinline__ Cpx<T> value_prod(const Cpx<T>* a, int2 k, int n) {
    Cpx<T> p = a[k.x & 0xffff];
    if (n > 1) p = cmul(p, a[(unsigned)k.x >> 16]);
    if (n > 2) p = cmul(p, a[k.y & 0xffff]);
    if (n > 3) p = cmul(p, a[(unsigned)k.y >> 16]);
    return p;
}

// ---------------------------------------------------------------------------
// Per atom: the derivatives of its energy E_i = sum_c c Pi x by the order parameters,
//   prod_sum_f[h] = 2 sum_f (dE_i / dx_f) (dx_f / da_h),
// and the energy from the same terms: with each column's coefficient divided by
// the number n_c of its order parameters (prod_sum_e),
//   E_i = sum_h w_h Re(a_h prod_sum_e[h]), w_h = 1/2 where m = 0. (The reference sums
// f_n Re(Y prod_sum_e) over pairs; an atom's sum of f_n Y is its a_h.)
// One workgroup of NL lanes (one wave, or four where there are few atoms or
// much work) per atom, the atom's order parameters, the features that the
// polynomial uses (its factors) and the columns' derivatives by them in LDS.
//   1. values of the factors;
//   2. dE/dx over the columns that hold a factor, each a coefficient times one
//      or two other factors (also with c / n_c), in pieces of equal length, a
//      lane each, added up in LDS;
//   3. per head, a lane: its terms, a coefficient (for features outside the
//      polynomial with dE/dx, a constant, folded in and merged), dE/dx and up
//      to three order parameters; heads in order of decreasing term count in
//      blocks of 64, so that a wave's lanes end together and no lane ends
//      inside another's head.
// Taking the gradient by the features first leaves about 600 terms instead of
// 11,792 for the one-type order-2 model (every column's derivative by every
// head before), and records of 12 or 16 bytes instead of 32: the tables come
// from L2 for every atom, which held the kernel at 8 TB/s on the 1,350-head
// model. FP64, 32,000 atoms of the one-type model: 0.71 -> 0.18 ms; 1,024-atom
// alloy: 0.40 -> 0.09 ms; 20,480 atoms of the alloy 1.49 ms.
// ---------------------------------------------------------------------------
template <class T, int NL>
__global__ void __launch_bounds__(NL) prodsum_kernel(ModelDev md, EvalDev ed, BatchDev bd,
                                                     const Cpx<T>* __restrict__ a_full,
                                                     int a_stride, Cpx<T>* __restrict__ ps_f,
                                                     Cpx<T>* __restrict__ ps_e, int ps_stride,
                                                     double* __restrict__ e_at, int pair_model) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    __shared__ double e_part[NL / 64];
    const int i = blockIdx.x;
    const int t1 = bd.types[i];
    const TypeDev& TT = md.t[t1];
    const EvalTypeDev& E = ed.t[t1];
    // sums of the derivatives by the factors; order parameters and the constant
    // 1; (derivatives, the same with c / n_c) by the factors, then the constants of features outside the polynomial with
    // 0 to 3 other order parameters; factors and 1
    using V2 = typename Vec2Of<T>::type;
    double2* sum = reinterpret_cast<double2*>(smem_raw);
    Cpx<T>* a = reinterpret_cast<Cpx<T>*>(sum + E.n_poly);
    V2* g = reinterpret_cast<V2*>(a + a_stride + 1);
    T* xs = reinterpret_cast<T*>(g + E.n_poly + 4);
    const int one = TT.n_nlm, lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr int NW = NL / 64;
    stage_cpx(a, a_full + (size_t)i * a_stride, TT.n_nlm);
    if (threadIdx.x == 0) a[one] = {T(1), T(0)}, xs[E.n_poly] = T(1);
    for (int q = threadIdx.x; q < E.n_poly; q += NL) sum[q] = E.pf_lin[q];
    if (threadIdx.x < 4) {
        V2 v;
        v.x = T(1), v.y = T(1) / T(int(threadIdx.x) + 1);
        g[E.n_poly + threadIdx.x] = v;
    }
    __syncthreads();
    {
        // products with |Re| <= 1e-20 are dropped where the reference drops them
        // (NaN is not one of them)
        const T least = TT.fv_skip ? T(1e-20) : T(-1);
        const T* c = EvalTab<T>::value(E);
        for (int bk = wave; bk < E.vq_nblk; bk += NW) {
            const int f = E.vq_item[bk * 64 + lane];
            T v = T(0);
            const int r1 = E.vq_boff[bk + 1];
#pragma unroll 2
            for (int r = E.vq_boff[bk] + lane; r < r1; r += 64) {
                const T p = value_prod<T>(a, E.vq_key[r], ed.value_max).re;
                v += fabs(p) <= least ? T(0) : c[r] * p;
            }
            if (f >= 0) xs[f] = v;
        }
    }
    __syncthreads();
    {
        const auto* c = EvalTab<T>::poly(E);
        for (int bk = wave; bk < E.pf_nblk; bk += NW) {
            const int r1 = E.pf_boff[bk + 1];
            double2 v = {0.0, 0.0};
#pragma unroll 4
            for (int r = E.pf_boff[bk] + lane; r < r1; r += 64) {
                const unsigned k = (unsigned)E.pf_rec[r];
                const double x = double(xs[k & 0xffff]) * double(xs[k >> 16]);
                const auto cr = c[r];
                v.x += double(cr.x) * x, v.y += double(cr.y) * x;
            }
            const int q = E.pf_piece[bk * 64 + lane];
            if (q >= 0) atomicAdd(&sum[q].x, v.x), atomicAdd(&sum[q].y, v.y);
        }
    }
    __syncthreads();
    for (int q = threadIdx.x; q < E.n_poly; q += NL) {
        V2 w;
        w.x = T(sum[q].x), w.y = T(sum[q].y);
        g[q] = w;
    }
    __syncthreads();
    const T scale = pair_model ? T(1) : T(2);
    double e_sum = 0.0;
    Cpx<T>* o = ps_f + (size_t)i * ps_stride;
    const T* c = EvalTab<T>::term(E);
    for (int bk = wave; bk < E.tq_nblk; bk += NW) {
        const int h = E.tq_item[bk * 64 + lane];
        T vr = T(0), vi = T(0), er = T(0), ei = T(0);
        const int r1 = E.tq_boff[bk + 1];
#pragma unroll 2
        for (int r = E.tq_boff[bk] + lane; r < r1; r += 64) {
            const int2 k = E.tq_key[r];
            const V2 w = g[(unsigned)k.y >> 16];
            const T cf = c[r] * w.x, ce = c[r] * w.y;
            Cpx<T> p = a[k.x & 0xffff];
            if (ed.term_max > 1) p = cmul(p, a[(unsigned)k.x >> 16]);
            if (ed.term_max > 2) p = cmul(p, a[k.y & 0xffff]);
            vr += cf * p.re, vi += cf * p.im;
            er += ce * p.re, ei += ce * p.im;
        }
        if (h >= 0) {
            o[h] = {scale * vr, scale * vi};
            if (ps_e) ps_e[(size_t)i * ps_stride + h] = {scale * er, scale * ei};
            const int ha = E.hd_a[h];  // the head's order parameter, bit 30: m = 0
            const Cpx<T> ac = a[ha & 0x3fffffff];
            const double v = double(er) * double(ac.re) - double(ei) * double(ac.im);
            e_sum += (ha >> 30) & 1 ? 0.5 * v : v;
        }
    }
    for (int off = 32; off > 0; off >>= 1) e_sum += __shfl_xor(e_sum, off);
    if (lane == 0) e_part[wave] = e_sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < NW; ++w) e_sum += e_part[w];
        e_at[i] = double(scale) * e_sum;
    }
}

// ---------------------------------------------------------------------------
// Half-pair loop, record form: one 64-lane workgroup per atom i. The records of up to
// kEvPairs of i's half pairs at a time (radial functions and derivatives,
// Y_lm and its gradient for the reversed vector r_i - r_j - T) are computed
// cooperatively in LDS (pairs_coop, the same arithmetic as the per-lane
// radial / ylm); then 8 lanes per pair split the pair's heads (lane slice s
// takes every 8th head) and the pair's sums are reduced over its 8 lanes.
// Nothing is indexed per lane at run time outside LDS, so no private arrays.
// ---------------------------------------------------------------------------
constexpr int kEvPairs = 8;  // pairs per chunk, 8 lanes each

template <class T>
__global__ void __launch_bounds__(64) pair_rec_kernel(ModelDev md, EvalDev ed, BatchDev bd,
                                                  const int* __restrict__ atom_st,
                                                  const int* __restrict__ hb_off,
                                                  const int* __restrict__ hb_j,
                                                  const double* __restrict__ hb_d,
                                                  const Cpx<T>* __restrict__ ps_f, int ps_stride,
                                                  double* __restrict__ forces,
                                                  double* __restrict__ stress, int pair_model) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    T* pairs = reinterpret_cast<T*>(smem_raw);
    const int i = blockIdx.x;
    if (i >= bd.n_atoms_total) return;
    const int p0 = hb_off[i], p1 = hb_off[i + 1];
    if (p0 == p1) return;
    const int t1 = bd.types[i];
    const EvalTypeDev& E = ed.t[t1];
    const PairLayout<T> L(md.n_fn, md.n_lmh);
    BatchDev hb = bd;  // the records are built from the half list
    hb.nb_j = hb_j;
    hb.nb_d = hb_d;
    const int lane = threadIdx.x, pl = lane >> 3, sl = lane & 7;
    const Cpx<T>* Pi_f = ps_f + (size_t)i * ps_stride;
    double fi_acc[3] = {0, 0, 0}, s_acc[6] = {0, 0, 0, 0, 0, 0};
    for (int c0 = p0; c0 < p1; c0 += kEvPairs) {
        const int np = min(kEvPairs, p1 - c0);
        __syncthreads();  // the previous chunk's records are read
        pairs_coop<T>(md, L, pairs, np, c0, hb, t1, 0, true, -1.0, pair_model ? -1 : md.max_l);
        const int k = c0 + pl;
        T* slot = pairs + (size_t)min(pl, np - 1) * L.stride;
        const T* ms = L.misc(slot);
        const bool live = pl < np && ms[4] != T(0);
        // pair model: fxa = radial-derivative sum
        T fxa = T(0), fya = T(0), fza = T(0);
        int j = 0;
        if (live) {
            const int tp = int(ms[5]);
            j = hb_j[k];
            const T* fn = L.fn(slot);
            const T* fd = L.fd(slot);
            const Cpx<T>* Pj_f = ps_f + (size_t)j * ps_stride;
            const int h0 = E.hd_off[tp], h1 = E.hd_off[tp + 1];
            if (pair_model) {
                for (int h = h0 + sl; h < h1; h += 8) {
                    const int4 hr = E.hd_rec[h];
                    const int nid = hr.x, hi = hr.z, hj = hr.w & 0x0fffffff;
                    fxa += fd[nid] * (Pi_f[hi].re + Pj_f[hj].re);
                }
            } else {
                const Cpx<T>* Y = L.Y(slot);
                const Cpx<T>* dY = L.dY(slot);
                const T dx = ms[0], dy = ms[1], dz = ms[2];
                const T ir = T(1) / ms[3];
                for (int h = h0 + sl; h < h1; h += 8) {
                    const int4 hr = E.hd_rec[h];
                    const int nid = hr.x;
                    const T fv = fn[nid];
                    if (fv < T(1e-20)) continue;
                    const int key = hr.y;
                    const int hi = hr.z, hj = hr.w & 0x0fffffff;
                    const T sj = (hr.w >> 28) & 1 ? T(-1) : T(1);
                    const T w = (hr.w >> 29) & 1 ? T(0.5) : T(1);
                    const Cpx<T> sf = {(Pi_f[hi].re + Pj_f[hj].re * sj) * w,
                                       (Pi_f[hi].im + Pj_f[hj].im * sj) * w};
                    const Cpx<T> y = Y[key];
                    const T d1r = fd[nid] * y.re * ir, d1i = fd[nid] * y.im * ir;
                    // val_a = -(d1 * d_a + fn * dY_a)
                    const Cpx<T> vx = {-(d1r * dx + fv * dY[3 * key].re), -(d1i * dx + fv * dY[3 * key].im)};
                    const Cpx<T> vy = {-(d1r * dy + fv * dY[3 * key + 1].re), -(d1i * dy + fv * dY[3 * key + 1].im)};
                    const Cpx<T> vz = {-(d1r * dz + fv * dY[3 * key + 2].re), -(d1i * dz + fv * dY[3 * key + 2].im)};
                    fxa += re_mul(vx, sf);
                    fya += re_mul(vy, sf);
                    fza += re_mul(vz, sf);
                }
            }
        }
        // the pair's sums over its 8 lanes
#pragma unroll
        for (int off = 1; off < 8; off <<= 1) {
            fxa += __shfl_xor(fxa, off);
            fya += __shfl_xor(fya, off);
            fza += __shfl_xor(fza, off);
        }
        if (live && sl == 0) {
            // diff_ij: r_i - r_j - T, in FP64 for the forces' directions and the stress
            const double dx = -hb_d[3 * (size_t)k], dy = -hb_d[3 * (size_t)k + 1],
                         dz = -hb_d[3 * (size_t)k + 2];
            double fx, fy, fz;
            if (pair_model) {
                const double fij = -double(fxa) / sqrt(dx * dx + dy * dy + dz * dz);
                fx = fij * dx, fy = fij * dy, fz = fij * dz;
            } else {
                fx = double(fxa), fy = double(fya), fz = double(fza);
            }
            fi_acc[0] += fx, fi_acc[1] += fy, fi_acc[2] += fz;
            atomicAdd(forces + 3 * (size_t)j, -fx);
            atomicAdd(forces + 3 * (size_t)j + 1, -fy);
            atomicAdd(forces + 3 * (size_t)j + 2, -fz);
            s_acc[0] += dx * fx, s_acc[1] += dy * fy, s_acc[2] += dz * fz;
            s_acc[3] += dx * fy, s_acc[4] += dy * fz, s_acc[5] += dz * fx;
        }
    }
    // wave reduction (64 lanes)
    for (int off = 32; off > 0; off >>= 1) {
        for (int a = 0; a < 3; ++a) fi_acc[a] += __shfl_down(fi_acc[a], off);
        for (int a = 0; a < 6; ++a) s_acc[a] += __shfl_down(s_acc[a], off);
    }
    if (lane == 0) {
        const int s = atom_st[i];
        for (int a = 0; a < 3; ++a) atomicAdd(forces + 3 * (size_t)i + a, fi_acc[a]);
        for (int a = 0; a < 6; ++a) atomicAdd(stress + 6 * (size_t)s + a, s_acc[a]);
    }
}

// ---------------------------------------------------------------------------
// Half-pair loop, per-lane form: one lane per half pair (i, j) of the whole
// list (bd carries the half list), Y_lm with its gradient generated column by
// column (LB bounds max l), each key used at once on its heads. The heads of a
// type pair are laid out by key, then by radial function, in the head sums of
// both atoms, so the heads of a key are two runs of cnt values, S_n = P_i[n] +
// (-1)^l P_j[n], and the force needs only A = sum_n f'_n S_n and B = sum_n f_n S_n:
//   f = -w (Re(Y A) d / r + Re(dY B)),  w = 1/2 where m = 0.
// f_n and f'_n sit in LDS, a column per lane (an array in registers, indexed
// by n, cost 48 KB of scratch a wave or a wave per SIMD). The forces on j go
// out as atomics per lane, those on i per run of lanes with the same i. A wave
// whose pairs belong to one structure writes its part of the stress to
// part[wave] (eval_sum_kernel adds the waves up): as atomics on the structure's
// six values the waves' sums took 13 ns each, one after the other, which was
// the kernel's whole time on one large cell (FP64, 32,000 atoms: 1.97 -> 0.40 ms;
// 160 alloys of 128 atoms 1.69 ms). blockIdx.y: the keys of m = y, y +
// gridDim.y, .. only (few pairs: more waves, each with part of the keys).
// ---------------------------------------------------------------------------
template <class T, int LB>
__global__ void __launch_bounds__(64) pair_lane_kernel(ModelDev md, EvalDev ed, BatchDev bd,
                                                   const int* __restrict__ atom_st,
                                                   int n_pairs,
                                                   const Cpx<T>* __restrict__ ps_f, int ps_stride,
                                                   double* __restrict__ forces,
                                                   double* __restrict__ stress,
                                                   double* __restrict__ part, int pair_model) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    using V2 = typename Vec2Of<T>::type;
    V2* rad = reinterpret_cast<V2*>(smem_raw);  // [n][lane]: f_n, f'_n
    const int lane = threadIdx.x;
    const int k = blockIdx.x * 64 + lane;
    double fx = 0.0, fy = 0.0, fz = 0.0;
    double dx = 0.0, dy = 0.0, dz = 0.0;
    int st = -1, i = -1, j = -1;
    if (k < n_pairs) {
        // atom i of pair k: nb_off[i] <= k < nb_off[i + 1]
        int lo = 0, hi = bd.n_atoms_total;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (bd.nb_off[mid] <= k) lo = mid;
            else hi = mid;
        }
        i = lo;
        st = atom_st[i];
        const int t1 = bd.types[i];
        const int jj = bd.nb_j[k];
        const int t2 = bd.types[jj];
        // diff_ij: r_i - r_j - T
        dx = -bd.nb_d[3 * (size_t)k], dy = -bd.nb_d[3 * (size_t)k + 1], dz = -bd.nb_d[3 * (size_t)k + 2];
        const double dis = sqrt(dx * dx + dy * dy + dz * dz);
        if (dis < md.cutoff) {
            j = jj;
            const int tp = md.tp_of[t1 * md.n_type + t2];
            const int cnt = md.rad_count[tp];
            // terms of f_n < 1e-20 are dropped (polymlp_eval.cpp:235)
            {
                const double* par = md.rad + (size_t)tp * md.n_fn * 2;
                const T r = T(dis), kc = MathConst<T>::pi / T(md.cutoff);
                T s, c;
                dsincos(kc * r, &s, &c);
                const T fc = T(0.5) * (c + T(1)), fcd = T(-0.5) * kc * s;
                for (int n = 0; n < (cnt + 3) / 4 * 4; ++n) {
                    const int nn = min(n, cnt - 1);
                    const T beta = T(par[2 * nn]), mu = T(par[2 * nn + 1]);
                    const T q = r - mu;
                    const T g = dexp(-beta * q * q);
                    const T gd = T(-2) * beta * q * g;
                    const T fv = g * fc;
                    const bool on = n < cnt && (pair_model || !(fv < T(1e-20)));
                    V2 v;
                    v.x = on ? fv : T(0), v.y = on ? gd * fc + g * fcd : T(0);
                    rad[64 * n + lane] = v;
                }
            }
            const V2* Pi = reinterpret_cast<const V2*>(ps_f + (size_t)i * ps_stride) + ed.t[t1].hd_off[tp];
            const V2* Pj = reinterpret_cast<const V2*>(ps_f + (size_t)j * ps_stride) + ed.t[t2].hd_off[tp];
            // A and B of the heads of key (rows of four radial functions, whose
            // last ones repeat the run's last value at zero weight)
            auto run = [&](int key, T sj, Cpx<T>& A, Cpx<T>& B) {
                const V2* pi = Pi + key * cnt;
                const V2* pj = Pj + key * cnt;
                A = {T(0), T(0)}, B = {T(0), T(0)};
                for (int n = 0; n < cnt; n += 4) {
                    V2 u[4], v[4], f[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q) u[q] = pi[min(n + q, cnt - 1)], v[q] = pj[min(n + q, cnt - 1)];
#pragma unroll
                    for (int q = 0; q < 4; ++q) f[q] = rad[64 * (n + q) + lane];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const T sr = u[q].x + sj * v[q].x, si = u[q].y + sj * v[q].y;
                        A.re += f[q].y * sr, A.im += f[q].y * si;
                        B.re += f[q].x * sr, B.im += f[q].x * si;
                    }
                }
            };
            if (pair_model) {
                Cpx<T> A, B;
                run(0, T(1), A, B);
                const double fij = -double(A.re) / dis;
                fx = fij * dx, fy = fij * dy, fz = fij * dz;
            } else {
                // Y_l^{-m} and its gradient generated column by column, m = max_l
                // down to 0 (column m needs Q(l, m + 1) of the column before), each
                // key used at once on its heads: the recurrences and operation
                // order of ylm(), with no array indexed at run time
                using C = MathConst<T>;
                const T x = T(dx), yy = T(dy), z = T(dz), r = T(dis);
                const T ct = z / r;
                const T rho = dhypot(x, yy);
                T cp = T(1), sp = T(0);
                if (rho > T(0)) cp = x / rho, sp = yy / rho;
                const T st = dsqrt(T(1) - ct * ct);
                const T invr = T(1) / r;
                const T ir = T(1) / T(dis);
                T cm[LB + 1], sm[LB + 1];  // cos, sin (m phi) by the Chebyshev recurrence
                cm[0] = T(1), sm[0] = T(0);
                {
                    T c1 = T(1), c2 = cp, s1 = T(0), s2 = -sp;
                    const T tc = T(2) * c2;
#pragma unroll
                    for (int mp = 1; mp <= LB; ++mp) {
                        const T sv = tc * s1 - s2;
                        const T cv = tc * c1 - c2;
                        c2 = c1, c1 = cv, s2 = s1, s1 = sv;
                        cm[mp] = cv, sm[mp] = sv;
                    }
                }
                const int lmax = md.max_l;
                T fxa = T(0), fya = T(0), fza = T(0);
                // l even or odd: the sign of the component seen from atom j
                auto heads = [&](int key, bool odd, T w, Cpx<T> y, Cpx<T> gx, Cpx<T> gy, Cpx<T> gz) {
                    Cpx<T> A, B;
                    run(key, odd ? T(-1) : T(1), A, B);
                    const T ra = re_mul(y, A) * ir;
                    fxa -= w * (ra * x + re_mul(gx, B));
                    fya -= w * (ra * yy + re_mul(gy, B));
                    fza -= w * (ra * z + re_mul(gz, B));
                };
                T qn[LB + 1];  // Q(l, m + 1)
#pragma unroll
                for (int l = 0; l <= LB; ++l) qn[l] = T(0);
#pragma unroll
                for (int m = LB; m >= 0; --m) {
                    if (m > lmax) continue;
                    // normalised associated Legendre column m: P and Q = P / sin(theta)
                    T pc[LB + 1], qc[LB + 1];
                    T pmm = C::sqrt_inv_2pi, qmm = T(0);
                    if (m >= 1) {
                        pmm = -st * C::sqrt3div2 * C::sqrt_inv_2pi;
                        qmm = -C::sqrt3div2 * C::sqrt_inv_2pi;
#pragma unroll
                        for (int l = 2; l <= m; ++l) {
                            const T c1 = -dsqrt(T(1) + T(0.5) / T(l)) * st;
                            pmm = c1 * pmm;
                            qmm = c1 * qmm;
                        }
                    }
#pragma unroll
                    for (int l = 0; l <= LB; ++l) pc[l] = T(0), qc[l] = T(0);
                    pc[m] = pmm, qc[m] = qmm;
                    if (m + 1 <= LB && m + 1 <= lmax) {
                        if (m == 0) {
                            pc[1] = ct * C::sqrt3 * C::sqrt_inv_2pi;
                            qc[1] = T(0);
                        } else {
                            const T c2 = dsqrt(T(2) * (T(m + 1) - T(1)) + T(3)) * ct;
                            pc[m + 1] = c2 * pmm;
                            qc[m + 1] = c2 * qmm;
                        }
#pragma unroll
                        for (int l = m + 2; l <= LB; ++l) {
                            if (l > lmax) break;
                            const T ls = T(l * l), lm1s = T((l - 1) * (l - 1)), msq = T(m * m);
                            const T alm = dsqrt((T(4) * ls - T(1)) / (ls - msq));
                            const T blm = -dsqrt((lm1s - msq) / (T(4) * lm1s - T(1)));
                            pc[l] = alm * (ct * pc[l - 1] + blm * pc[l - 2]);
                            qc[l] = alm * (ct * qc[l - 1] + blm * qc[l - 2]);
                        }
                    }
#pragma unroll
                    for (int l = m; l <= LB; ++l) {
                        if (l > lmax || m % (int)gridDim.y != (int)blockIdx.y) break;
                        if (m == 0) {
                            const T common =
                                (l >= 1) ? qn[l] * st * invr * dsqrt(T(0.5) * T(l) * T(l + 1)) : T(0);
                            heads(lm2i(l, 0) + l, l & 1, T(0.5), Cpx<T>{pc[l] * C::half_sqrt2, T(0)},
                                  Cpx<T>{common * ct * cp, T(0)}, Cpx<T>{common * ct * sp, T(0)},
                                  Cpx<T>{-common * st, T(0)});
                        } else {
                            const T c = cm[m], sv = sm[m];
                            const T sign = (m % 2 == 1) ? T(-1) : T(1);
                            const T tmp = sign * pc[l] * C::half_sqrt2;
                            const T cre = c * C::half_sqrt2 * invr, cim = sv * C::half_sqrt2 * invr;
                            T dth = T(m) * ct * qc[l];
                            if (m != l) dth += dsqrt(T((l - m) * (l + m + 1))) * qn[l] * st;
                            const T dph = T(m) * qc[l];
                            const T ure = dth * ct * cp, uim = -dph * sp;
                            const T vre = dth * ct * sp, vim = dph * cp;
                            const T wre = -dth * st;
                            heads(lm2i(l, -m) + l, l & 1, T(1), Cpx<T>{tmp * c, -tmp * sv},
                                  Cpx<T>{sign * (cre * ure - cim * uim), -sign * (cre * uim + cim * ure)},
                                  Cpx<T>{sign * (cre * vre - cim * vim), -sign * (cre * vim + cim * vre)},
                                  Cpx<T>{sign * (cre * wre), -sign * (cim * wre)});
                        }
                    }
#pragma unroll
                    for (int l = 0; l <= LB; ++l) qn[l] = qc[l];
                }
                fx = double(fxa), fy = double(fya), fz = double(fza);
            }
        }
    }
    if (j >= 0) {
        atomicAdd(forces + 3 * (size_t)j, -fx);
        atomicAdd(forces + 3 * (size_t)j + 1, -fy);
        atomicAdd(forces + 3 * (size_t)j + 2, -fz);
    }
    // the lanes of one i are neighbours: the first of them gets their sum
    double si[3] = {fx, fy, fz};
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int io = __shfl_down(i, off);
        const bool same = lane + off < 64 && io == i;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const double v = __shfl_down(si[a], off);
            if (same) si[a] += v;
        }
    }
    const int ip = __shfl_up(i, 1);
    if (i >= 0 && (lane == 0 || ip != i))
        for (int a = 0; a < 3; ++a) atomicAdd(forces + 3 * (size_t)i + a, si[a]);
    double sv[6] = {dx * fx, dy * fy, dz * fz, dx * fy, dy * fz, dz * fx};
    const int s0 = __builtin_amdgcn_readfirstlane(st);
    if (__all(st == s0 || st < 0)) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1)
#pragma unroll
            for (int a = 0; a < 6; ++a) sv[a] += __shfl_down(sv[a], off);
        if (lane == 0)
            for (int a = 0; a < 6; ++a)
                part[6 * ((size_t)blockIdx.y * gridDim.x + blockIdx.x) + a] = sv[a];
    } else if (st >= 0) {
        for (int a = 0; a < 6; ++a) atomicAdd(stress + 6 * (size_t)st + a, sv[a]);
    }
}

// Per structure: its atoms' energies, and the stress parts of the pair loop's
// waves that lie whole in its pairs (parts rows of n_waves; null: none).
__global__ void __launch_bounds__(256) eval_sum_kernel(BatchDev bd, int n_pairs, int n_waves,
                                                       int parts, const double* __restrict__ part,
                                                       const double* __restrict__ e_at,
                                                       double* __restrict__ energy,
                                                       double* __restrict__ stress) {
    __shared__ double sum[7][4];
    const int s = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int a0 = bd.st_atom_off[s], a1 = bd.st_atom_off[s + 1];
    const int step = 256 * gridDim.y, first = 256 * blockIdx.y + threadIdx.x;
    double v[7] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
    for (int i = a0 + first; i < a1; i += step) v[6] += e_at[i];
    if (part) {
        const int h0 = bd.nb_off[a0], h1 = bd.nb_off[a1];
        const int w0 = (h0 + 63) / 64, w1 = h1 == n_pairs ? n_waves : h1 / 64;
        for (int y = 0; y < parts; ++y) {
            const double* p = part + 6 * (size_t)y * n_waves;
#pragma unroll 2
            for (int w = w0 + first; w < w1; w += step)
#pragma unroll
                for (int a = 0; a < 6; ++a) v[a] += p[6 * (size_t)w + a];
        }
    }
#pragma unroll
    for (int a = 0; a < 7; ++a) {
        for (int off = 32; off > 0; off >>= 1) v[a] += __shfl_down(v[a], off);
        if (lane == 0) sum[a][wave] = v[a];
    }
    __syncthreads();
    if (threadIdx.x < 7) {
        const int a = threadIdx.x;
        const double t = (sum[a][0] + sum[a][1]) + (sum[a][2] + sum[a][3]);
        double* o = a < 6 ? stress + 6 * (size_t)s + a : energy + s;
        if (gridDim.y == 1) *o += t;
        else atomicAdd(o, t);
    }
}

static size_t prodsum_smem(const EvalDev& ed, int a_stride, size_t elem) {
    return (size_t)ed.poly_max * sizeof(double2) + (size_t)(a_stride + 1) * 2 * elem +
           (size_t)(ed.poly_max + 4) * 2 * elem + (size_t)(ed.poly_max + 1) * elem;
}

// dynamic LDS of a workgroup, next to the waves' energies
static constexpr size_t kProdsumLds = 160 * 1024 - 64;

bool prodsum_fits(const EvalDev& ed, bool fp64, int a_stride) {
    return prodsum_smem(ed, a_stride, fp64 ? 8 : 4) <= kProdsumLds;
}

template <class T, int NL>
void launch_prodsum_t(hipStream_t st, const ModelDev& md, const EvalDev& ed, const BatchDev& bd,
                      const void* a_full, int a_stride, void* ps_f, void* ps_e, int ps_stride,
                      double* e_at, int pair_model) {
    const size_t sm = prodsum_smem(ed, a_stride, sizeof(T));
    if (sm > kProdsumLds) throw std::invalid_argument("per-atom evaluation data exceed LDS");
    check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(&prodsum_kernel<T, NL>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)sm),
              "prodsum shared memory");
    prodsum_kernel<T, NL><<<bd.n_atoms_total, NL, sm, st>>>(
        md, ed, bd, reinterpret_cast<const Cpx<T>*>(a_full), a_stride,
        reinterpret_cast<Cpx<T>*>(ps_f), reinterpret_cast<Cpx<T>*>(ps_e), ps_stride, e_at,
        pair_model);
}

// Four waves an atom where its table rows are more than 128 or the atoms do
// not fill the chip with eight waves a SIMD, else one (FP64, 20,480 atoms of the
// 1,350-head model: 1.49 ms with four, 4.74 with one; 54 atoms of the one-type
// model 11 and 17 us; 32,000 atoms of it 0.184 and 0.171 ms);
// PLM_PRODSUM_LANES=64|256 forces one form.
void launch_prodsum(hipStream_t st, bool fp64, const ModelDev& md, const EvalDev& ed,
                    const BatchDev& bd, const void* a_full, int a_stride, void* ps_f,
                    void* ps_e, int ps_stride, double* e_at, int pair_model) {
    bool four = ed.rows_max > 128 || bd.n_atoms_total < 8192;
    if (const char* e = std::getenv("PLM_PRODSUM_LANES")) {
        if (!std::strcmp(e, "64")) four = false;
        else if (!std::strcmp(e, "256")) four = true;
        else throw std::invalid_argument("PLM_PRODSUM_LANES must be 64 or 256");
    }
    if (fp64 && four)
        launch_prodsum_t<double, 256>(st, md, ed, bd, a_full, a_stride, ps_f, ps_e, ps_stride,
                                      e_at, pair_model);
    else if (fp64)
        launch_prodsum_t<double, 64>(st, md, ed, bd, a_full, a_stride, ps_f, ps_e, ps_stride,
                                     e_at, pair_model);
    else if (four)
        launch_prodsum_t<float, 256>(st, md, ed, bd, a_full, a_stride, ps_f, ps_e, ps_stride,
                                     e_at, pair_model);
    else
        launch_prodsum_t<float, 64>(st, md, ed, bd, a_full, a_stride, ps_f, ps_e, ps_stride,
                                    e_at, pair_model);
}

template <class T>
void launch_pair_rec_t(hipStream_t st, const ModelDev& md, const EvalDev& ed, const BatchDev& bd,
                   const int* atom_st, const void* ps_f, int ps_stride, double* forces,
                   double* stress, int pair_model) {
    const size_t sm = (size_t)kEvPairs * PairLayout<T>(md.n_fn, md.n_lmh).stride * sizeof(T);
    if (sm > 160 * 1024) throw std::invalid_argument("evaluation pair records exceed LDS");
    check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(&pair_rec_kernel<T>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)sm),
              "pair shared memory");
    pair_rec_kernel<T><<<bd.n_atoms_total, 64, sm, st>>>(
        md, ed, bd, atom_st, bd.nb_off, bd.nb_j, bd.nb_d, reinterpret_cast<const Cpx<T>*>(ps_f),
        ps_stride, forces, stress, pair_model);
}

// Waves of the per-lane form and the parts its keys are split into: with fewer
// waves than two a SIMD, the keys of a pair are dealt by m to several (54 atoms:
// 21 waves; 138 us with all keys in one lane, 44 us so).
static int pair_parts(const ModelDev& md, int waves, int pair_model) {
    return pair_model ? 1 : std::max(1, std::min(md.max_l + 1, (2048 + waves - 1) / waves));
}

template <class T, int LB>
void launch_pair_lb(hipStream_t st, const ModelDev& md, const EvalDev& ed, const BatchDev& bd,
                    const int* atom_st, int n_half, const void* ps_f, int ps_stride,
                    double* forces, double* stress, double* part, int pair_model) {
    const int waves = (n_half + 63) / 64;
    const size_t sm = (size_t)((md.n_fn + 3) / 4 * 4) * 64 * 2 * sizeof(T);
    pair_lane_kernel<T, LB><<<dim3(waves, pair_parts(md, waves, pair_model)), 64, sm, st>>>(
        md, ed, bd, atom_st, n_half, reinterpret_cast<const Cpx<T>*>(ps_f), ps_stride, forces,
        stress, part, pair_model);
}

template <class T>
void launch_pair_lane_t(hipStream_t st, const ModelDev& md, const EvalDev& ed,
                        const BatchDev& bd, const int* atom_st, int n_half, const void* ps_f,
                        int ps_stride, double* forces, double* stress, double* part,
                        int pair_model) {
    const int L = md.max_l;
    if (md.n_fn > 32)
        throw std::invalid_argument("the per-lane pair loop supports at most 32 radial functions");
    if (L <= 4)
        launch_pair_lb<T, 4>(st, md, ed, bd, atom_st, n_half, ps_f, ps_stride, forces, stress,
                             part, pair_model);
    else if (L <= 8)
        launch_pair_lb<T, 8>(st, md, ed, bd, atom_st, n_half, ps_f, ps_stride, forces, stress,
                             part, pair_model);
    else if (L <= 12)
        launch_pair_lb<T, 12>(st, md, ed, bd, atom_st, n_half, ps_f, ps_stride, forces, stress,
                              part, pair_model);
    else
        throw std::invalid_argument("the per-lane pair loop supports max_l <= 12");
}

size_t pair_part_bytes(const ModelDev& md, int n_half, int pair_model) {
    const int waves = (std::max(n_half, 1) + 63) / 64;
    return (size_t)waves * pair_parts(md, waves, pair_model) * 48;
}

// The per-lane form where it applies (max_l <= 12, at most 32 radial
// functions), the record form beyond; PLM_EVAL_PAIR=lane / records forces one.
// e_at: the atoms' energies (launch_prodsum), added up per structure here.
void launch_pair(hipStream_t st, bool fp64, const ModelDev& md, const EvalDev& ed,
                 const BatchDev& bd, const int* atom_st, int n_half, const double* e_at,
                 const void* ps_f, int ps_stride, double* part, double* energy, double* forces,
                 double* stress, int pair_model) {
    if (n_half <= 0) return;
    bool lane = md.max_l <= 12 && md.n_fn <= 32;
    if (const char* e = getenv("PLM_EVAL_PAIR")) {
        if (!strcmp(e, "lane")) lane = true;
        else if (!strcmp(e, "records")) lane = false;
        else throw std::invalid_argument("PLM_EVAL_PAIR: lane or records");
    }
    if (lane && fp64)
        launch_pair_lane_t<double>(st, md, ed, bd, atom_st, n_half, ps_f, ps_stride, forces,
                                   stress, part, pair_model);
    else if (lane)
        launch_pair_lane_t<float>(st, md, ed, bd, atom_st, n_half, ps_f, ps_stride, forces, stress,
                                  part, pair_model);
    else if (fp64)
        launch_pair_rec_t<double>(st, md, ed, bd, atom_st, ps_f, ps_stride, forces, stress,
                                  pair_model);
    else
        launch_pair_rec_t<float>(st, md, ed, bd, atom_st, ps_f, ps_stride, forces, stress,
                                 pair_model);
    // a workgroup per structure, several for structures of more than 4,096 waves
    const int waves = (n_half + 63) / 64, parts = pair_parts(md, waves, pair_model);
    const int split = std::max(1, std::min(16, waves * parts / bd.n_st / 2048));
    eval_sum_kernel<<<dim3(bd.n_st, split), 256, 0, st>>>(bd, n_half, waves, parts,
                                                          lane ? part : nullptr, e_at, energy,
                                                          stress);
}

__global__ void __launch_bounds__(256) fill_zero_kernel(double* __restrict__ x, size_t n) {
    for (size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x; k < n;
         k += (size_t)gridDim.x * blockDim.x)
        x[k] = 0.0;
}

void launch_fill_zero(hipStream_t st, double* x, size_t n) {
    if (n == 0) return;
    const size_t blocks = std::min<size_t>((n + 255) / 256, 4096);
    fill_zero_kernel<<<(unsigned)blocks, 256, 0, st>>>(x, n);
}

}  // namespace plm
