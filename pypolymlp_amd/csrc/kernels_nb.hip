// Neighbour lists with the reference's pair sets, order and rounding.
//
// A pair (i, j, T) is kept by the reference's distance predicate evaluated
// with the same rounded FP64 operations as NeighborFull (neighbor_full.cpp:10-76;
// no FMA contraction), and each atom's list is in the reference's order, (j,
// translation index) ascending, so the lists are bit-identical. Two searches:
// every (j, T) of the structure, and for one large cell a cell list (bins).
//
// The half list of the evaluation (NeighborHalf, neighbor_half.cpp:10-100) is
// the full list's entries with j < i, followed by the self images in the upper
// half space of the translation: the same predicate on the same operands, so
// it is filtered from the full list instead of searched again.
#include <hip/hip_runtime.h>

#include <stdexcept>

#include "kernels.hpp"

namespace plm {

// d = (r_j - r_i) + T, kept when tol2 < |d|^2 < cut2
__device__ __forceinline__ bool in_range(double dxij, double dyij, double dzij, const double* tr,
                                         double cut2, double tol2, double* d) {
    const double dx = __dadd_rn(dxij, tr[0]);
    const double dy = __dadd_rn(dyij, tr[1]);
    const double dz = __dadd_rn(dzij, tr[2]);
    const double r2 = __dadd_rn(__dadd_rn(__dmul_rn(dx, dx), __dmul_rn(dy, dy)), __dmul_rn(dz, dz));
    d[0] = dx, d[1] = dy, d[2] = dz;
    return r2 < cut2 && r2 > tol2;
}

// upper half space of a self image's translation (neighbor_half.cpp:55-76)
__device__ __forceinline__ bool upper_half(double dx, double dy, double dz, double tol) {
    return dz >= tol || (fabs(dz) < tol && dy >= tol) ||
           (fabs(dz) < tol && fabs(dy) < tol && dx >= tol);
}

__device__ __forceinline__ int wave_sum(int v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

__device__ __forceinline__ int wave_inclusive(int v, int lane) {
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int u = __shfl_up(v, off);
        if (lane >= off) v += u;
    }
    return v;
}

// start[k] = sum of count[< k], start[n] = the total, for the counts of
// workgroup blockIdx.x (n each); clear: the counts become zero
__global__ void __launch_bounds__(1024) scan_kernel(int n, int* __restrict__ count,
                                                    int* __restrict__ start, int clear) {
    __shared__ int part[16];
    count += (size_t)n * blockIdx.x, start += (size_t)(n + 1) * blockIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int base = 0;
    for (int k0 = 0; k0 < n; k0 += 4096) {
        const int k = k0 + 4 * threadIdx.x;
        int c[4], sum = 0;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            c[u] = k + u < n ? count[k + u] : 0;
            sum += c[u];
        }
        const int incl = wave_inclusive(sum, lane);
        if (lane == 63) part[wave] = incl;
        __syncthreads();
        int out = base + incl - sum, all = 0;
        for (int w = 0; w < 16; ++w) {
            if (w < wave) out += part[w];
            all += part[w];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (k + u < n) {
                start[k + u] = out;
                if (clear) count[k + u] = 0;
                out += c[u];
            }
        base += all;
        __syncthreads();
    }
    if (threadIdx.x == 0) start[n] = base;
}

// ---------------------------------------------------------------------------
// All (j, T) of the structure. One workgroup per atom i (a wave per 64 atoms
// of its structure, at most four), one lane per j: the difference r_j - r_i is
// formed once and the translations are the same for every lane, so they come
// through scalar loads and a candidate costs nine FP64 operations.
// Bound by those operations. (One thread per atom, before, left a 1024-atom
// cell on 16 waves: 4.4 ms a pass and four passes; evaluating that cell went
// from 19.8 to 1.6 ms, a 54-atom cell from 1.89 to 0.34 ms.)
// ---------------------------------------------------------------------------
constexpr int kListThreads = 256;

// count[i]: full list, count[n + i]: half list
__global__ void __launch_bounds__(kListThreads) list_count_kernel(
    int n, const int* __restrict__ atom_st, const int* __restrict__ st_atom_off,
    const double* __restrict__ pos, const int* __restrict__ tr_off,
    const double* __restrict__ trans, double cut2, double tol2, double tol,
    int* __restrict__ count) {
    __shared__ int part[2][kListThreads / 64];
    const int i = blockIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int s = atom_st[i];
    const int a0 = st_atom_off[s], a1 = st_atom_off[s + 1];
    const int t0 = tr_off[s], t1 = tr_off[s + 1];
    const double px = pos[3 * (size_t)i], py = pos[3 * (size_t)i + 1], pz = pos[3 * (size_t)i + 2];
    int full = 0, half = 0;
    for (int j = a0 + threadIdx.x; j < a1; j += blockDim.x) {
        const double* pj = pos + 3 * (size_t)j;
        const double dx = __dadd_rn(pj[0], -px), dy = __dadd_rn(pj[1], -py),
                     dz = __dadd_rn(pj[2], -pz);
        int c = 0;
        for (int t = t0; t < t1; ++t) {
            double d[3];
            c += in_range(dx, dy, dz, trans + 3 * (size_t)t, cut2, tol2, d) ? 1 : 0;
        }
        full += c;
        if (j < i) half += c;
    }
    for (int t = t0 + threadIdx.x; t < t1; t += blockDim.x) {
        const double* tr = trans + 3 * (size_t)t;
        double d[3];
        if (in_range(0.0, 0.0, 0.0, tr, cut2, tol2, d) && upper_half(tr[0], tr[1], tr[2], tol)) ++half;
    }
    full = wave_sum(full), half = wave_sum(half);
    if (lane == 0) part[0][wave] = full, part[1][wave] = half;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < (int)(blockDim.x >> 6); ++w) full += part[0][w], half += part[1][w];
        count[i] = full;
        count[n + i] = half;
    }
}

// The full list. j ascends over the lanes, then over the waves, then over the
// rounds of a workgroup, so a lane's place is the prefix sum of the counts
// before it. Up to 128 translations a lane keeps the hits as bits and forms
// only the kept pairs again; beyond, it searches a second time.
template <bool BITS>
__global__ void __launch_bounds__(kListThreads) list_fill_kernel(
    const int* __restrict__ atom_st, const int* __restrict__ st_atom_off,
    const double* __restrict__ pos, const int* __restrict__ tr_off,
    const double* __restrict__ trans, double cut2, double tol2, const int* __restrict__ nb_off,
    int* __restrict__ nb_j, int* __restrict__ nb_t, double* __restrict__ nb_d) {
    __shared__ int part[kListThreads / 64];
    const int i = blockIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const int s = atom_st[i];
    const int a0 = st_atom_off[s], a1 = st_atom_off[s + 1];
    const int t0 = tr_off[s], t1 = tr_off[s + 1];
    const double px = pos[3 * (size_t)i], py = pos[3 * (size_t)i + 1], pz = pos[3 * (size_t)i + 2];
    int base = nb_off[i];
    for (int jb = a0; jb < a1; jb += blockDim.x) {
        const int j = jb + threadIdx.x;
        double dx = 0.0, dy = 0.0, dz = 0.0;
        unsigned bits[4] = {0u, 0u, 0u, 0u};
        int c = 0;
        if (j < a1) {
            const double* pj = pos + 3 * (size_t)j;
            dx = __dadd_rn(pj[0], -px), dy = __dadd_rn(pj[1], -py), dz = __dadd_rn(pj[2], -pz);
            double d[3];
            if constexpr (BITS) {
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const int tb = t0 + 32 * w, te = min(t1, tb + 32);
                    for (int t = tb; t < te; ++t)
                        if (in_range(dx, dy, dz, trans + 3 * (size_t)t, cut2, tol2, d))
                            bits[w] |= 1u << (t - tb);
                    c += __popc(bits[w]);
                }
            } else {
                for (int t = t0; t < t1; ++t)
                    c += in_range(dx, dy, dz, trans + 3 * (size_t)t, cut2, tol2, d) ? 1 : 0;
            }
        }
        const int incl = wave_inclusive(c, lane);
        if (lane == 63) part[wave] = incl;
        __syncthreads();
        int out = base + incl - c, all = 0;
        for (int w = 0; w < nw; ++w) {
            if (w < wave) out += part[w];
            all += part[w];
        }
        auto emit = [&](int t) {
            double d[3];
            if (!in_range(dx, dy, dz, trans + 3 * (size_t)t, cut2, tol2, d)) return;
            nb_j[out] = j;
            nb_t[out] = t - t0;
            double* o = nb_d + 3 * (size_t)out;
            o[0] = d[0], o[1] = d[1], o[2] = d[2];
            ++out;
        };
        if (c > 0) {
            if constexpr (BITS) {
#pragma unroll
                for (int w = 0; w < 4; ++w)
                    for (unsigned b = bits[w]; b; b &= b - 1) emit(t0 + 32 * w + __ffs(b) - 1);
            } else {
                for (int t = t0; t < t1; ++t) emit(t);
            }
        }
        base += all;
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// Cell list for one large cell. Atoms are binned on their wrapped fractional
// coordinates. For atom i and each of the 27 neighbouring bins, an image of
// atom j is the integer lattice shift k = s - w_j + w_i (s: bin wrap, w: floor
// of the fractional coordinates); the pair is a candidate only if k is one of
// the reference's lattice translations (NeighborCell::find_trans,
// neighbor_cell.cpp:236-255).
// ---------------------------------------------------------------------------
struct BinGrid {
    int nb[3];
    int mexp[3];          // translation index box: k_a in [-mexp_a, mexp_a]
    double inv[9];        // inverse of the axis used for translations (row-major)
    const int* tindex;    // [(2m0+1)(2m1+1)(2m2+1)] -> translation index or -1
};

// an atom in bin order
struct __attribute__((aligned(16))) BinAtom {
    double r[3];
    int w[3];  // wraps
    int j;
};

__global__ void bin_assign_kernel(int n, const double* __restrict__ pos, BinGrid g,
                                  int* __restrict__ bin, int* __restrict__ wrap,
                                  int* __restrict__ bin_count) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double* r = pos + 3 * (size_t)i;
    int b[3];
    for (int a = 0; a < 3; ++a) {
        const double f = g.inv[3 * a] * r[0] + g.inv[3 * a + 1] * r[1] + g.inv[3 * a + 2] * r[2];
        const double w = floor(f);
        const double fw = f - w;
        int bb = (int)(fw * g.nb[a]);
        bb = min(max(bb, 0), g.nb[a] - 1);
        b[a] = bb;
        wrap[3 * (size_t)i + a] = (int)w;
    }
    const int id = (b[0] * g.nb[1] + b[1]) * g.nb[2] + b[2];
    bin[i] = id;
    atomicAdd(bin_count + id, 1);
}

__global__ void bin_scatter_kernel(int n, const int* __restrict__ bin, const int* __restrict__ start,
                                   const double* __restrict__ pos, const int* __restrict__ wrap,
                                   int* __restrict__ cursor, BinAtom* __restrict__ sorted) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int b = bin[i];
    BinAtom a;
    for (int k = 0; k < 3; ++k) a.r[k] = pos[3 * (size_t)i + k], a.w[k] = wrap[3 * (size_t)i + k];
    a.j = i;
    sorted[start[b] + atomicAdd(cursor + b, 1)] = a;
}

// One wave per atom, lanes over the atoms of the 27 bins laid end to end (a
// lane finds its bin by a search in the bins' prefix sums). FILL: the kept
// (j, translation) keys go to LDS (GKEYS: to global memory, where an atom has
// more neighbours than LDS holds), each entry's place is the number of smaller
// keys, and the kept pairs' differences are formed again from the keys.
// Bound by the latency of the candidates' loads; a wave has about five rounds
// of them (one thread per atom with an insertion sort in memory took 27
// dependent rounds: 0.95 ms a pass on 32,000 atoms, 11 ms on 2,744 atoms where
// three bins span the cell; evaluating those went from 8.0 to 4.6 and from 41.7
// to 1.0 ms).
template <bool FILL, bool GKEYS>
__global__ void __launch_bounds__(64) bin_pairs_kernel(
    int n, const double* __restrict__ pos, const int* __restrict__ bin,
    const int* __restrict__ start, const BinAtom* __restrict__ sorted, BinGrid g,
    const double* __restrict__ trans, double cut2, double tol2, double tol,
    int* __restrict__ count, const int* __restrict__ nb_off, int* __restrict__ nb_j,
    int* __restrict__ nb_t, double* __restrict__ nb_d, unsigned long long* __restrict__ gkeys) {
    __shared__ int pre[28], first[27], kx[27], ky[27], kz[27];
    extern __shared__ unsigned long long lkeys[];
    const int lane = threadIdx.x;
    const BinAtom me = sorted[blockIdx.x];
    const int i = me.j;
    {
        int len = 0;
        if (lane < 27) {
            const int bi = bin[i];
            const int b[3] = {bi / (g.nb[1] * g.nb[2]), (bi / g.nb[2]) % g.nb[1], bi % g.nb[2]};
            const int o[3] = {lane / 9 - 1, lane / 3 % 3 - 1, lane % 3 - 1};
            int c[3], sh[3];
            for (int a = 0; a < 3; ++a) {
                const int q = b[a] + o[a];
                sh[a] = q < 0 ? -1 : (q >= g.nb[a] ? 1 : 0);
                c[a] = q - sh[a] * g.nb[a];
            }
            const int cb = (c[0] * g.nb[1] + c[1]) * g.nb[2] + c[2];
            first[lane] = start[cb];
            len = start[cb + 1] - first[lane];
            kx[lane] = sh[0] + me.w[0], ky[lane] = sh[1] + me.w[1], kz[lane] = sh[2] + me.w[2];
        }
        const int incl = wave_inclusive(len, lane);
        if (lane < 28) pre[lane] = incl - len;  // lane 27: the total
    }
    __syncthreads();
    const int total = pre[27];
    const int M1 = 2 * g.mexp[1] + 1, M2 = 2 * g.mexp[2] + 1;
    const int out0 = FILL ? nb_off[i] : 0;
    unsigned long long* keys = GKEYS ? gkeys + out0 : lkeys;
    int full = 0, half = 0;
    for (int e0 = 0; e0 < total; e0 += 64) {
        const int e = e0 + lane;
        bool keep = false;
        int j = 0, t = -1;
        if (e < total) {
            int b = 0;
#pragma unroll
            for (int st = 16; st > 0; st >>= 1)
                if (b + st < 27 && pre[b + st] <= e) b += st;
            const BinAtom q = sorted[first[b] + e - pre[b]];
            j = q.j;
            const int k0 = kx[b] - q.w[0], k1 = ky[b] - q.w[1], k2 = kz[b] - q.w[2];
            if (k0 >= -g.mexp[0] && k0 <= g.mexp[0] && k1 >= -g.mexp[1] && k1 <= g.mexp[1] &&
                k2 >= -g.mexp[2] && k2 <= g.mexp[2]) {
                t = g.tindex[((k0 + g.mexp[0]) * M1 + (k1 + g.mexp[1])) * M2 + (k2 + g.mexp[2])];
                if (t >= 0) {
                    const double* tr = trans + 3 * (size_t)t;
                    double d[3];
                    keep = in_range(__dadd_rn(q.r[0], -me.r[0]), __dadd_rn(q.r[1], -me.r[1]),
                                    __dadd_rn(q.r[2], -me.r[2]), tr, cut2, tol2, d);
                    if (!FILL && keep && (j < i || (j == i && upper_half(tr[0], tr[1], tr[2], tol))))
                        ++half;
                }
            }
        }
        const unsigned long long vote = __ballot(keep);
        if (FILL && keep)
            keys[full + __popcll(vote & ((1ull << lane) - 1ull))] =
                (unsigned long long)(unsigned)j << 32 | (unsigned)t;
        full += __popcll(vote);
    }
    if (!FILL) {
        half = wave_sum(half);
        if (lane == 0) count[i] = full, count[n + i] = half;
        return;
    }
    __syncthreads();
    for (int e = lane; e < full; e += 64) {
        const unsigned long long key = keys[e];
        int o = out0;
        for (int q = 0; q < full; ++q) o += keys[q] < key ? 1 : 0;
        const int j = (int)(key >> 32), t = (int)(key & 0xffffffffull);
        const double* pj = pos + 3 * (size_t)j;
        double d[3];
        (void)in_range(__dadd_rn(pj[0], -me.r[0]), __dadd_rn(pj[1], -me.r[1]),
                       __dadd_rn(pj[2], -me.r[2]), trans + 3 * (size_t)t, cut2, tol2, d);
        nb_j[o] = j;
        nb_t[o] = t;
        double* od = nb_d + 3 * (size_t)o;
        od[0] = d[0], od[1] = d[1], od[2] = d[2];
    }
}

// ---------------------------------------------------------------------------
// The half list from the full one: one wave per atom, kept entries in order.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) half_list_kernel(
    int n, double tol, const int* __restrict__ nb_off, const int* __restrict__ nb_j,
    const int* __restrict__ nb_t, const double* __restrict__ nb_d, const int* __restrict__ hb_off,
    int* __restrict__ hb_j, int* __restrict__ hb_t, double* __restrict__ hb_d) {
    const int i = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (i >= n) return;
    int out = hb_off[i];
    const int p1 = nb_off[i + 1];
    for (int p0 = nb_off[i]; p0 < p1; p0 += 64) {
        const int p = p0 + lane;
        bool keep = false;
        int j = n;
        double d[3] = {0.0, 0.0, 0.0};
        if (p < p1) {
            j = nb_j[p];
            for (int a = 0; a < 3; ++a) d[a] = nb_d[3 * (size_t)p + a];
            keep = j < i || (j == i && upper_half(d[0], d[1], d[2], tol));
        }
        const unsigned long long vote = __ballot(keep);
        if (keep) {
            const int o = out + __popcll(vote & ((1ull << lane) - 1ull));
            hb_j[o] = j;
            if (hb_t) hb_t[o] = nb_t[p];
            for (int a = 0; a < 3; ++a) hb_d[3 * (size_t)o + a] = d[a];
        }
        out += __popcll(vote);
        if (__all(j > i)) break;  // j ascends
    }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
static int list_threads(int max_atoms) {
    return 64 * (max_atoms > 192 ? 4 : (max_atoms + 63) / 64);
}

void launch_list_count(hipStream_t st, int n, int max_atoms, const int* atom_st,
                       const int* st_atom_off, const double* pos, const int* tr_off,
                       const double* trans, double cut2, double tol2, double tol, int* count) {
    list_count_kernel<<<n, list_threads(max_atoms), 0, st>>>(n, atom_st, st_atom_off, pos, tr_off,
                                                             trans, cut2, tol2, tol, count);
}

void launch_list_fill(hipStream_t st, int n, int max_atoms, int max_trans, const int* atom_st,
                      const int* st_atom_off, const double* pos, const int* tr_off,
                      const double* trans, double cut2, double tol2, const int* nb_off, int* nb_j,
                      int* nb_t, double* nb_d) {
    // the hits of 128 translations fit four words a lane
    if (max_trans <= 128)
        list_fill_kernel<true><<<n, list_threads(max_atoms), 0, st>>>(
            atom_st, st_atom_off, pos, tr_off, trans, cut2, tol2, nb_off, nb_j, nb_t, nb_d);
    else
        list_fill_kernel<false><<<n, list_threads(max_atoms), 0, st>>>(
            atom_st, st_atom_off, pos, tr_off, trans, cut2, tol2, nb_off, nb_j, nb_t, nb_d);
}

void launch_list_offsets(hipStream_t st, int n, int* count, int* off) {
    scan_kernel<<<2, 1024, 0, st>>>(n, count, off, 0);
}

static BinGrid device_grid(const BinGridHost& gh) {
    BinGrid g;
    for (int a = 0; a < 3; ++a) g.nb[a] = gh.nb[a], g.mexp[a] = gh.mexp[a];
    for (int a = 0; a < 9; ++a) g.inv[a] = gh.inv[a];
    g.tindex = gh.tindex;
    return g;
}

size_t bin_atom_bytes() { return sizeof(BinAtom); }

void launch_bin_atoms(hipStream_t st, int n, const double* pos, const BinGridHost& gh, int* bin,
                      int* wrap, int* bin_count, int* start, void* sorted) {
    const int nbins = gh.nb[0] * gh.nb[1] * gh.nb[2];
    bin_assign_kernel<<<(n + 255) / 256, 256, 0, st>>>(n, pos, device_grid(gh), bin, wrap, bin_count);
    scan_kernel<<<1, 1024, 0, st>>>(nbins, bin_count, start, 1);  // the counts become cursors
    bin_scatter_kernel<<<(n + 255) / 256, 256, 0, st>>>(n, bin, start, pos, wrap, bin_count,
                                                        static_cast<BinAtom*>(sorted));
}

void launch_bin_count(hipStream_t st, int n, const double* pos, const int* bin, const int* start,
                      const void* sorted, const BinGridHost& gh, const double* trans, double cut2,
                      double tol2, double tol, int* count) {
    bin_pairs_kernel<false, false><<<n, 64, 0, st>>>(
        n, pos, bin, start, static_cast<const BinAtom*>(sorted), device_grid(gh), trans, cut2, tol2,
        tol, count, nullptr, nullptr, nullptr, nullptr, nullptr);
}

// sort keys in LDS up to this many neighbours an atom (16 KB a wave, so LDS
// still leaves ten waves a CU); denser cells sort through global memory
constexpr int kLdsKeys = 2048;

size_t bin_key_bytes(long n_pairs, int max_pairs_atom) {
    return max_pairs_atom <= kLdsKeys ? 0 : (size_t)n_pairs * 8;
}

void launch_bin_fill(hipStream_t st, int n, int max_pairs_atom, const double* pos, const int* bin,
                     const int* start, const void* sorted, const BinGridHost& gh,
                     const double* trans, double cut2, double tol2, double tol, const int* nb_off,
                     int* nb_j, int* nb_t, double* nb_d, void* keys) {
    const BinAtom* sa = static_cast<const BinAtom*>(sorted);
    if (keys) {
        bin_pairs_kernel<true, true><<<n, 64, 0, st>>>(
            n, pos, bin, start, sa, device_grid(gh), trans, cut2, tol2, tol, nullptr, nb_off, nb_j,
            nb_t, nb_d, static_cast<unsigned long long*>(keys));
        return;
    }
    if (max_pairs_atom > kLdsKeys) throw std::invalid_argument("cell-list keys exceed LDS");
    const size_t sm = (size_t)max_pairs_atom * 8;
    bin_pairs_kernel<true, false><<<n, 64, sm, st>>>(n, pos, bin, start, sa, device_grid(gh), trans,
                                                     cut2, tol2, tol, nullptr, nb_off, nb_j, nb_t,
                                                     nb_d, nullptr);
}

void launch_half_list(hipStream_t st, int n, double tol, const int* nb_off, const int* nb_j,
                      const int* nb_t, const double* nb_d, const int* hb_off, int* hb_j, int* hb_t,
                      double* hb_d) {
    half_list_kernel<<<(n + 3) / 4, 256, 0, st>>>(n, tol, nb_off, nb_j, nb_t, nb_d, hb_off, hb_j,
                                                  hb_t, hb_d);
}

}  // namespace plm
