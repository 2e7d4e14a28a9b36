// Device tables of the potential used by evaluation.
#pragma once

#include "device_tables.hpp"

namespace plm {

struct EvalTypeDev {
    int n_heads;            // non-conjugate components (gtinv) or pair components
    // The features that columns of two and three features use, the polynomial's
    // factors. Their value terms, in blocks of 64 factors (one per lane), term
    // j of lane l at row j; keys of up to four order parameters, 16 bits each,
    // absent ones at the constant n_nlm:
    int n_poly;
    int vq_nblk;
    const int* vq_boff;
    const int* vq_item;
    const int2* vq_key;
    const double* vq_c;
    const float* vq_cf;
    // and the columns that hold factor q, in pieces (of factor pf_piece, -1
    // past the end) in blocks of 64 (one per lane), column j of lane l at row j: the other
    // factors o1 | o2 << 16 (o2 = n_poly, the constant 1, for columns of two)
    // and the column's coefficient times the factor's power, and that over the
    // number of the column's order parameters; pf_lin: both of the factor's linear
    // column
    int pf_nblk;
    const int* pf_boff;
    const int* pf_piece;
    const int* pf_rec;
    const double2* pf_c;
    const float2* pf_cf;
    const double2* pf_lin;
    // The terms of d x_f / d a_h, heads (by position) in order of decreasing
    // term count, in blocks of 64 (one per lane), term j of lane l at row j as
    // TypeDev's value terms: keys (pd0 | pd1 << 16, pd2 | factor << 16; absent
    // order parameters point at the constant n_nlm, features outside the
    // polynomial at factor n_poly + their number, the column's coefficient folded in)
    int tq_nblk;
    const int* tq_boff;
    const int* tq_item;
    const int2* tq_key;
    const double* tq_c;
    const float* tq_cf;
    // per head, its order parameter (index into the atom's full list) with bit
    // 30 set where m == 0
    const int* hd_a;
    // half-pair contraction: heads of this type grouped by type pair
    const int* hd_off;      // [n_tp+1]
    // gtinv: the heads of each type pair are ordered by Y key, then by radial
    // function (head hd_off[tp] + key * rad_count[tp] + n_id), in both atoms' head sums
    // per head, one 16-byte record: (radial n_id, ylm key, ilocal_noconj of the
    // head (atom i), jlocal_noconj (the same component seen from atom j) with
    // bit 28 set where (-1)^l = -1 and bit 29 where m == 0 (weight 1/2))
    const int4* hd_rec;
};

struct EvalDev {
    EvalTypeDev t[kMaxTypes];
    int value_max;          // order parameters of a value term, at most
    int term_max;           // order parameters of a derivative term, at most
    int poly_max;           // factors of a type, at most
    int rows_max;           // table rows of an atom's contraction, at most
};

}  // namespace plm
