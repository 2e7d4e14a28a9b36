// Evaluation (PolymlpEval) orchestration: potential tables (Potential,
// polymlp_potential.cpp:25-156; the factor 2 of polymlp_eval.cpp:12-20 is in the
// contraction), half neighbour list, order parameters, per-atom prod_sum and the
// half-pair loop.
#include <algorithm>
#include <array>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <numeric>
#include <stdexcept>
#include <vector>

#include "capi_internal.hpp"
#include "profile.hpp"

namespace plm {

namespace {

// Host tables of one potential, laid end to end, uploaded by one copy (about 20
// small arrays a type: one by one they cost 10 us each, most of set_coeffs for a
// small model).
struct TableUpload {
    std::vector<unsigned char> data;
    std::vector<std::pair<size_t, std::function<void(const unsigned char*)>>> set;
    template <class V>
    void put(const V*& dst, const std::vector<V>& v) {
        const size_t at = (data.size() + 63) / 64 * 64;
        data.resize(at + std::max<size_t>(1, v.size()) * sizeof(V));
        if (!v.empty()) std::memcpy(data.data() + at, v.data(), v.size() * sizeof(V));
        set.push_back({at, [&dst](const unsigned char* p) { dst = reinterpret_cast<const V*>(p); }});
    }
    void upload(Store& store) {
        const unsigned char* base = store.upload(data.data(), data.size());
        for (auto& s : set) s.second(base + s.first);
    }
};

}  // namespace

void upload_potential(ModelHandle& m) {
    const Model& M = m.host;
    if (!M.has_potential()) throw std::runtime_error("coefficients not set");
    m.pot_store.bufs.clear();
    m.pot_uploaded = false;
    TableUpload tables;
    const int nt = M.n_type(), ntp = M.n_tp();
    const bool gt = M.input().gtinv;
    m.max_heads = 0;
    m.ed.value_max = std::max(1, m.v_maxf), m.ed.term_max = 1;
    m.ed.poly_max = 0, m.ed.rows_max = 0;
    // The heads of each type in the order of the half-pair loop: grouped by type
    // pair, within one ordered by Y key (the per-lane pair loop generates Y_lm
    // key by key). The contraction writes head k of an atom at its position
    // rank[t][k] in that order, so the pair loop reads both atoms' sums in
    // address order. Entries: (radial n_id, ylm key, head k, head seen from
    // atom j, sign, m == 0).
    using HeadEntry = std::array<int, 6>;
    std::vector<std::vector<std::vector<HeadEntry>>> by_tp_t(nt);
    std::vector<std::vector<int>> order(nt);
    m.head_rank.assign(nt, {});
    for (int t = 0; t < nt; ++t) {
        const auto& T = M.type(t);
        auto& by_tp = by_tp_t[t];
        by_tp.assign(ntp, {});
        if (gt) {
            for (size_t k = 0; k < T.noconj.size(); ++k) {
                const auto& a = T.nlm[T.noconj[k]];
                by_tp[a.tp].push_back({a.n_id, a.ylm_key, (int)k, a.jlocal_noconj,
                                       a.sign_j < 0 ? -1 : 1, a.m == 0 ? 1 : 0});
            }
        } else {
            for (size_t k = 0; k < T.ntp.size(); ++k)
                by_tp[T.ntp[k][2]].push_back({T.ntp[k][1], -1, (int)k, T.ntp[k][3], 1, 0});
        }
        const int n_heads = (int)(gt ? T.noconj.size() : T.ntp.size());
        auto& rank = m.head_rank[t];
        rank.assign(n_heads, -1);
        for (int tp = 0; tp < ntp; ++tp) {
            if (gt)
                std::stable_sort(by_tp[tp].begin(), by_tp[tp].end(),
                                 [](const HeadEntry& a, const HeadEntry& b) { return a[1] < b[1]; });
            for (const auto& e : by_tp[tp]) {
                if (e[2] < 0 || e[2] >= n_heads || rank[e[2]] >= 0)
                    throw std::invalid_argument("evaluation heads do not match the potential");
                rank[e[2]] = (int)order[t].size();
                order[t].push_back(e[2]);
            }
        }
        if ((int)order[t].size() != n_heads)
            throw std::invalid_argument("evaluation heads do not match the potential");
    }
    // the first head position of each type pair
    std::vector<std::vector<int>> tp_first(nt, std::vector<int>(ntp, 0));
    for (int t = 0; t < nt; ++t)
        for (int tp = 1; tp < ntp; ++tp)
            tp_first[t][tp] = tp_first[t][tp - 1] + (int)by_tp_t[t][tp - 1].size();
    // the type of atom j for an atom of type t and a type pair
    auto partner = [&](int t, int tp) {
        int found = -1;
        for (int t2 = 0; t2 < nt; ++t2)
            if (M.type_pair(t, t2) == tp) {
                if (found >= 0) throw std::invalid_argument("type pair with two partner types");
                found = t2;
            }
        return found;
    };
    for (int t = 0; t < nt; ++t) {
        const auto& T = M.type(t);
        EvalTypeDev& E = m.ed.t[t];
        E.n_heads = (int)order[t].size();
        m.max_heads = std::max(m.max_heads, E.n_heads);
        // per type pair its heads; hi and hj are head positions of atoms i and j
        const int nkey = m.md.n_lmh;
        std::vector<int> hoff(ntp + 1, 0), nid, ylm, hi, hj;
        std::vector<float> sj;
        std::vector<unsigned char> m0;
        for (int tp = 0; tp < ntp; ++tp) {
            const auto& heads = by_tp_t[t][tp];
            const int t2 = heads.empty() ? -1 : partner(t, tp);
            if (!heads.empty() && t2 < 0) throw std::invalid_argument("type pair without partner type");
            for (const auto& e : heads) {
                if (gt && (e[1] < 0 || e[1] >= nkey)) throw std::invalid_argument("head Y key range");
                if (e[3] < 0 || e[3] >= (int)m.head_rank[t2].size())
                    throw std::invalid_argument("head of atom j out of range");
                nid.push_back(e[0]), ylm.push_back(e[1]);
                hi.push_back(m.head_rank[t][e[2]]), hj.push_back(m.head_rank[t2][e[3]]);
                sj.push_back((float)e[4]), m0.push_back((unsigned char)e[5]);
            }
            hoff[tp + 1] = (int)nid.size();
            // the layout the per-lane pair loop relies on
            const int cnt = (int)M.tp_to_n()[tp].size(), n_tp_heads = hoff[tp + 1] - hoff[tp];
            if (n_tp_heads != 0 && n_tp_heads != (gt ? nkey : 1) * cnt)
                throw std::invalid_argument("evaluation heads of a type pair");
            for (int h = hoff[tp]; h < hoff[tp + 1]; ++h)
                if (hi[h] != h || hj[h] - hj[hoff[tp]] != h - hoff[tp] ||
                    nid[h] != (h - hoff[tp]) % cnt || (gt && ylm[h] != (h - hoff[tp]) / cnt) ||
                    hj[hoff[tp]] != tp_first[t2][tp])
                    throw std::invalid_argument("evaluation head order");
        }
        auto k16 = [](int v) -> unsigned {
            if (v < 0 || v >= 0xffff) throw std::invalid_argument("evaluation table index exceeds 16 bits");
            return (unsigned)v;
        };
        const std::vector<double>& coef = M.coeffs();
        const int n_lin = (int)T.features.size();
        const unsigned none = k16(m.md.t[t].n_nlm);
        std::vector<double> lin(std::max(1, n_lin), 0.0);
        std::vector<int> factor(std::max(1, n_lin), -1), pf_feat;
        for (const auto& p : T.poly) {
            if (p.local_ids.size() == 1) {
                lin[p.local_ids[0]] += coef[p.global_id];
                continue;
            }
            if (p.local_ids.size() > 3) throw std::invalid_argument("polynomial order above 3");
            for (int f : p.local_ids)
                if (factor[f] < 0) factor[f] = (int)pf_feat.size(), pf_feat.push_back(f);
        }
        E.n_poly = (int)pf_feat.size();
        m.ed.poly_max = std::max(m.ed.poly_max, E.n_poly);
        struct PolyRec {
            unsigned rec;
            double2 c;
        };
        auto order_of = [&](int f) { return (int)T.features[f][0].ids.size(); };
        std::vector<std::vector<PolyRec>> by_factor(E.n_poly);
        for (const auto& p : T.poly) {
            const auto& id = p.local_ids;
            if (id.size() == 1) continue;
            int n_prods = 0;
            for (int f : id) n_prods += order_of(f);
            // each distinct factor once, with its power as a coefficient
            for (size_t q = 0; q < id.size(); ++q) {
                if (std::find(id.begin(), id.begin() + q, id[q]) != id.begin() + q) continue;
                const int power = (int)std::count(id.begin(), id.end(), id[q]);
                std::vector<int> o;
                for (size_t r = 0; r < id.size(); ++r)
                    if (r != q) o.push_back(factor[id[r]]);
                const double c = power * coef[p.global_id];
                by_factor[factor[id[q]]].push_back(
                    {k16(o[0]) | k16(o.size() > 1 ? o[1] : E.n_poly) << 16, double2{c, c / n_prods}});
            }
        }
        // pieces of at most `len` columns: the smallest that leaves 256 of them (a
        // block for each of four waves), or whole multiples for more factors
        size_t len = 8;
        const size_t most = (size_t)std::max(1, (E.n_poly + 255) / 256) * 256;
        for (;; ++len) {
            size_t n = 0;
            for (const auto& v : by_factor) n += (v.size() + len - 1) / len;
            if (n <= most) break;
        }
        std::vector<std::pair<int, size_t>> pieces;  // factor, first column
        std::vector<double2> pf_lin;
        for (int q = 0; q < E.n_poly; ++q) {
            for (size_t r = 0; r < by_factor[q].size(); r += len) pieces.push_back({q, r});
            const int f = pf_feat[q];
            pf_lin.push_back(double2{lin[f], lin[f] / order_of(f)});
        }
        E.pf_nblk = (int)(pieces.size() + 63) / 64;
        std::vector<int> pf_piece((size_t)E.pf_nblk * 64, -1);
        for (size_t p = 0; p < pieces.size(); ++p) pf_piece[p] = pieces[p].first;
        std::vector<int> pf_boff(E.pf_nblk + 1, 0), pf_rec;
        std::vector<double2> pf_c;
        for (int bk = 0; bk < E.pf_nblk; ++bk) {
            auto size_of = [&](size_t p) {
                return std::min(len, by_factor[pieces[p].first].size() - pieces[p].second);
            };
            const size_t p1 = std::min(pieces.size(), (size_t)(bk + 1) * 64);
            size_t rows = 0;
            for (size_t p = (size_t)bk * 64; p < p1; ++p) rows = std::max(rows, size_of(p));
            pf_boff[bk + 1] = pf_boff[bk] + (int)rows * 64;
            pf_rec.resize(pf_boff[bk + 1], (int)(k16(E.n_poly) | k16(E.n_poly) << 16));
            pf_c.resize(pf_boff[bk + 1], double2{0.0, 0.0});
            for (size_t p = (size_t)bk * 64; p < p1; ++p)
                for (size_t j = 0; j < size_of(p); ++j) {
                    const PolyRec& v = by_factor[pieces[p].first][pieces[p].second + j];
                    const size_t r = (size_t)pf_boff[bk] + j * 64 + (p - (size_t)bk * 64);
                    pf_rec[r] = (int)v.rec, pf_c[r] = v.c;
                }
        }
        // the factors' value terms
        auto value_key = [&](int prod) {
            const auto& k = T.prod[prod];
            if (k.size() > 4) throw std::invalid_argument("invariant order above 4");
            unsigned p[4] = {none, none, none, none};
            for (size_t q = 0; q < k.size(); ++q) p[q] = k16(k[q]);
            return int2{(int)(p[0] | p[1] << 16), (int)(p[2] | p[3] << 16)};
        };
        std::vector<int> vq(E.n_poly);
        std::iota(vq.begin(), vq.end(), 0);
        std::stable_sort(vq.begin(), vq.end(), [&](int x, int y) {
            return T.feat_val[pf_feat[x]].size() > T.feat_val[pf_feat[y]].size();
        });
        E.vq_nblk = (E.n_poly + 63) / 64;
        std::vector<int> vboff(E.vq_nblk + 1, 0), vitem((size_t)E.vq_nblk * 64, -1);
        std::vector<int2> vkey;
        std::vector<double> vc;
        for (int bk = 0; bk < E.vq_nblk; ++bk) {
            vboff[bk + 1] = vboff[bk] + (int)T.feat_val[pf_feat[vq[bk * 64]]].size() * 64;
            vkey.resize(vboff[bk + 1], int2{(int)(none | none << 16), (int)(none | none << 16)});
            vc.resize(vboff[bk + 1], 0.0);
            for (int l = 0; l < 64 && bk * 64 + l < E.n_poly; ++l) {
                const int q = vq[bk * 64 + l];
                vitem[(size_t)bk * 64 + l] = q;
                size_t r = (size_t)vboff[bk] + l;
                for (const auto& pc : T.feat_val[pf_feat[q]])
                    vkey[r] = value_key(pc.first), vc[r] = pc.second, r += 64;
            }
        }
        // derivative terms by head position; terms of one product and factor are
        // one (features outside the polynomial share the constant factor)
        struct Term {
            int prod, factor;
            double c;
        };
        std::vector<std::vector<Term>> terms(E.n_heads);
        for (int f = 0; f < n_lin; ++f)
            for (const auto& d : T.feat_deriv[f]) {
                if (gt && T.nlm[d.head].conj) continue;
                const int k = gt ? T.local_to_noconj[d.head] : d.head;
                const bool poly = factor[f] >= 0;
                const int n_pd = (int)T.prod_deriv[d.prod].size();
                if (n_pd > 3) throw std::invalid_argument("term order too high");
                terms[m.head_rank[t][k]].push_back(
                    {d.prod, poly ? factor[f] : E.n_poly + n_pd, poly ? d.coeff : d.coeff * lin[f]});
            }
        for (auto& v : terms) {
            std::stable_sort(v.begin(), v.end(), [](const Term& x, const Term& y) {
                return x.prod != y.prod ? x.prod < y.prod : x.factor < y.factor;
            });
            size_t n = 0;
            for (size_t q = 0; q < v.size(); ++q)
                if (n > 0 && v[n - 1].prod == v[q].prod && v[n - 1].factor == v[q].factor)
                    v[n - 1].c += v[q].c;
                else
                    v[n++] = v[q];
            v.resize(n);
        }
        std::vector<int> by_count(E.n_heads);
        std::iota(by_count.begin(), by_count.end(), 0);
        std::stable_sort(by_count.begin(), by_count.end(),
                         [&](int x, int y) { return terms[x].size() > terms[y].size(); });
        E.tq_nblk = (E.n_heads + 63) / 64;
        const unsigned pad_y = none | k16(E.n_poly) << 16;
        std::vector<int> boff(E.tq_nblk + 1, 0), item((size_t)E.tq_nblk * 64, -1);
        std::vector<int2> key;
        std::vector<double> tc;
        for (int bk = 0; bk < E.tq_nblk; ++bk) {
            const int rows = (int)terms[by_count[bk * 64]].size();
            boff[bk + 1] = boff[bk] + rows * 64;
            key.resize(boff[bk + 1], int2{(int)(none | none << 16), (int)pad_y});
            tc.resize(boff[bk + 1], 0.0);
            for (int l = 0; l < 64 && bk * 64 + l < E.n_heads; ++l) {
                const int h = by_count[bk * 64 + l];
                item[(size_t)bk * 64 + l] = h;
                for (size_t j = 0; j < terms[h].size(); ++j) {
                    const auto& pd = T.prod_deriv[terms[h][j].prod];
                    m.ed.term_max = std::max(m.ed.term_max, (int)pd.size());
                    unsigned p[3] = {none, none, none};
                    for (size_t q = 0; q < pd.size(); ++q) p[q] = k16(pd[q]);
                    const size_t r = (size_t)boff[bk] + j * 64 + l;
                    key[r] = int2{(int)(p[0] | p[1] << 16), (int)(p[2] | k16(terms[h][j].factor) << 16)};
                    tc[r] = terms[h][j].c;
                }
            }
        }
        m.ed.rows_max = std::max<int>(m.ed.rows_max, (boff[E.tq_nblk] + vboff[E.vq_nblk] +
                                                      (int)pf_rec.size()) / 64);
        const std::vector<float> tcf(tc.begin(), tc.end()), vcf(vc.begin(), vc.end());
        std::vector<float2> pf_cf;
        for (const double2& c : pf_c) pf_cf.push_back(float2{(float)c.x, (float)c.y});
        std::vector<int> ha(std::max(1, E.n_heads), 0);
        for (int r = 0; r < E.n_heads; ++r) {
            const int k = order[t][r];
            ha[r] = gt ? T.noconj[k] | (T.nlm[T.noconj[k]].m == 0 ? 1 << 30 : 0) : k;
        }
        tables.put(E.hd_a, ha);
        tables.put(E.vq_boff, vboff), tables.put(E.vq_item, vitem), tables.put(E.vq_key, vkey);
        tables.put(E.vq_c, vc), tables.put(E.vq_cf, vcf);
        tables.put(E.pf_boff, pf_boff), tables.put(E.pf_piece, pf_piece);
        tables.put(E.pf_rec, pf_rec), tables.put(E.pf_lin, pf_lin);
        tables.put(E.pf_c, pf_c), tables.put(E.pf_cf, pf_cf);
        tables.put(E.tq_boff, boff), tables.put(E.tq_item, item), tables.put(E.tq_key, key);
        tables.put(E.tq_c, tc), tables.put(E.tq_cf, tcf);
        std::vector<int4> rec(std::max<size_t>(1, nid.size()), int4{0, 0, 0, 0});
        for (size_t h = 0; h < nid.size(); ++h) {
            if (hj[h] < 0 || hj[h] >= (1 << 28)) throw std::invalid_argument("head index range");
            rec[h] = int4{nid[h], ylm[h], hi[h],
                          hj[h] | (sj[h] < 0.f ? 1 << 28 : 0) | (m0[h] ? 1 << 29 : 0)};
        }
        tables.put(E.hd_off, hoff), tables.put(E.hd_rec, rec);
    }
    tables.upload(m.pot_store);
    m.pot_uploaded = true;
    ++m.pot_version;
}

bool eval_in_fp64(const ModelHandle& m, bool fp64) {
    return fp64 || (anlm_fits(m.md, true, m.max_noconj) && prodsum_fits(m.ed, true, m.max_nlm));
}

// Work buffers of one evaluation; out = [energies | forces (3 per atom) | stresses (6)].
static void alloc_eval(const ModelHandle& m, const BatchHandle& b, bool fp64, DevBuf& a_buf,
                       DevBuf& e_at, DevBuf& psf, DevBuf& part, DevBuf& out, size_t& n_out) {
    const int elem = fp64 ? 8 : 4;
    const size_t A = b.n_atoms;
    a_buf.alloc(A * m.max_nlm * 2 * elem);
    e_at.alloc(A * 8);
    part.alloc(pair_part_bytes(m.md, (int)b.n_half, m.host.input().gtinv ? 0 : 1));
    psf.alloc(A * std::max(1, m.max_heads) * 2 * elem);
    n_out = (size_t)b.n_st + 3 * A + 6 * (size_t)b.n_st;
    out.alloc(n_out * 8);
}

// The kernels of one evaluation on st: out is cleared by a kernel (no memset
// node when captured), then filled by the half-pair loop. bd carries the full
// neighbour list (order parameters); hb_* the half list (pair loop).
void enqueue_eval_dev(ModelHandle& m, const BatchDev& bd, const int* hb_off, const int* hb_j,
                      const double* hb_d, int n_half, bool fp64, void* a_buf, double* e_at,
                      void* psf, double* part, double* out, size_t n_out, hipStream_t st) {
    const int A = bd.n_atoms_total;
    launch_fill_zero(st, out, n_out);
    double* d_e = out;
    double* d_f = d_e + bd.n_st;
    double* d_s = d_f + 3 * (size_t)A;
    const int pair_model = m.host.input().gtinv ? 0 : 1;
    {
        ProfScope ps("eval_anlm", st);
        launch_anlm(st, fp64, m.md, bd, a_buf, m.max_nlm, 0, A, m.max_noconj, 1);
    }
    check_hip(hipGetLastError(), "eval anlm launch");
    {
        ProfScope ps("eval_prodsum", st);
        launch_prodsum(st, fp64, m.md, m.ed, bd, a_buf, m.max_nlm, psf, nullptr,
                       std::max(1, m.max_heads), e_at, pair_model);
    }
    check_hip(hipGetLastError(), "prodsum launch");
    {
        ProfScope ps("eval_pair", st);
        BatchDev hb = bd;
        hb.nb_off = hb_off, hb.nb_j = hb_j, hb.nb_d = hb_d;
        launch_pair(st, fp64, m.md, m.ed, hb, bd.atom_st, n_half, e_at, psf,
                    std::max(1, m.max_heads), part, d_e, d_f, d_s, pair_model);
    }
    check_hip(hipGetLastError(), "pair launch");
}

static void enqueue_eval(ModelHandle& m, BatchHandle& b, bool fp64, void* a_buf, double* e_at,
                         void* psf, double* part, double* out, size_t n_out, hipStream_t st) {
    enqueue_eval_dev(m, b.view(), b.d_hb_off(), (const int*)b.d_hb_j.ptr,
                     (const double*)b.d_hb_d.ptr, (int)b.n_half, fp64, a_buf, e_at, psf, part, out,
                     n_out, st);
}

// h: staging on the host (kept by the caller, so that its pages are in place)
static void copy_out(const BatchHandle& b, const DevBuf& out, size_t n_out, hipStream_t st,
                     std::vector<double>& h, double* energies, double* forces, double* stresses) {
    const size_t A = b.n_atoms;
    if (h.size() < n_out) h.resize(n_out);
    check_hip(hipMemcpyAsync(h.data(), out.ptr, n_out * 8, hipMemcpyDeviceToHost, st), "copy");
    check_hip(hipStreamSynchronize(st), "sync");
    if (energies) std::memcpy(energies, h.data(), (size_t)b.n_st * 8);
    if (forces) std::memcpy(forces, h.data() + b.n_st, 3 * A * 8);
    if (stresses) std::memcpy(stresses, h.data() + b.n_st + 3 * A, 6 * (size_t)b.n_st * 8);
}

static void prepare_eval(ModelHandle& m, BatchHandle& b) {
    if (!m.built) m.build_device();
    if (!m.pot_uploaded) upload_potential(m);
    b.ensure_half();
}

void eval_batch(ModelHandle& m, BatchHandle& b, bool fp64, double* energies, double* forces,
                double* stresses) {
    prepare_eval(m, b);
    fp64 = eval_in_fp64(m, fp64);
    hipStream_t st = device().stream;
    std::lock_guard<std::mutex> lock(m.eval_mutex);
    size_t n_out = 0;
    alloc_eval(m, b, fp64, m.ev_a, m.ev_eat, m.ev_psf, m.ev_part, m.ev_out, n_out);
    enqueue_eval(m, b, fp64, m.ev_a.ptr, (double*)m.ev_eat.ptr, m.ev_psf.ptr, (double*)m.ev_part.ptr, (double*)m.ev_out.ptr, n_out,
                 st);
    copy_out(b, m.ev_out, n_out, st, m.ev_host, energies, forces, stresses);
}

EvalGraph::~EvalGraph() {
    if (exec) (void)hipGraphExecDestroy(exec);
    if (graph) (void)hipGraphDestroy(graph);
}

void eval_graph_capture(EvalGraph& g) {
    ModelHandle& m = *g.m;
    BatchHandle& b = *g.b;
    prepare_eval(m, b);
    g.fp64 = eval_in_fp64(m, g.fp64);
    hipStream_t st = device().stream;
    alloc_eval(m, b, g.fp64, g.a_buf, g.e_at, g.psf, g.part, g.out, g.n_out);
    // one eager pass first: kernel attributes are set and every buffer exists
    enqueue_eval(m, b, g.fp64, g.a_buf.ptr, (double*)g.e_at.ptr, g.psf.ptr, (double*)g.part.ptr, (double*)g.out.ptr, g.n_out, st);
    check_hip(hipStreamSynchronize(st), "sync");
    {
        ProfPause pause;
        check_hip(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal), "begin capture");
        try {
            enqueue_eval(m, b, g.fp64, g.a_buf.ptr, (double*)g.e_at.ptr, g.psf.ptr, (double*)g.part.ptr, (double*)g.out.ptr,
                         g.n_out, st);
        } catch (...) {
            hipGraph_t tmp = nullptr;
            (void)hipStreamEndCapture(st, &tmp);
            if (tmp) (void)hipGraphDestroy(tmp);
            throw;
        }
        check_hip(hipStreamEndCapture(st, &g.graph), "end capture");
    }
    check_hip(hipGraphInstantiate(&g.exec, g.graph, nullptr, nullptr, 0), "graph instantiate");
    g.pot_version = m.pot_version;
}

void eval_graph_run(EvalGraph& g, int steps, double* energies, double* forces, double* stresses) {
    if (steps < 1) throw std::invalid_argument("steps must be positive");
    if (!g.m->pot_uploaded || g.m->pot_version != g.pot_version)
        throw std::invalid_argument("model coefficients changed since the graph was captured");
    hipStream_t st = device().stream;
    for (int k = 0; k < steps; ++k) check_hip(hipGraphLaunch(g.exec, st), "graph launch");
    std::vector<double> h;
    copy_out(*g.b, g.out, g.n_out, st, h, energies, forces, stresses);
}

void eval_single(ModelHandle& m, const double* axis, const double* pos_c, const int* types, int n,
                 bool fp64, double* energy, double* forces, double* stress) {
    if (!m.built) m.build_device();
    BatchHandle b(&m, m.host.input().cutoff, 1, axis, pos_c, types, &n);
    eval_batch(m, b, fp64, energy, forces, stress);
}

}  // namespace plm
