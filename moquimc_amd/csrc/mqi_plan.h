// Host-side planning of the sparse products, as plain functions (no HIP), so
// they are testable on any host.
#ifndef MQI_PLAN_H
#define MQI_PLAN_H

#include <stddef.h>
#include <stdint.h>

#include <algorithm>
#include <vector>

// Pieces of the D^T g product over column deltas (each at most 65535 within
// a piece): each row of a CSR
// (row pointers ip[0..rows]) is cut at its first nonzero, at every position
// in `gaps` (ascending; nonzeros whose column is more than 65535 past the
// previous one of the row; positions at a row start are ignored) and every
// `plen` nonzeros after a cut; an empty row gets one empty piece (the product
// writes every row through its pieces).  pk receives the first nonzero of
// each piece in order plus the sentinel ip[rows]; row_piece[r] (rows + 1
// entries) the first piece of row r.  Returns false when the pieces would not
// fit int32.
static inline bool
cut_pieces(const std::vector<int64_t>& ip, const std::vector<int64_t>& gaps, int64_t plen,
           std::vector<int64_t>& pk, std::vector<int32_t>& row_piece) {
    const int64_t rows = (int64_t) ip.size() - 1;
    pk.clear();
    row_piece.assign((size_t) rows + 1, 0);
    if (plen < 1) plen = 1;
    size_t gi = 0;
    for (int64_t i = 0; i < rows; ++i) {
        row_piece[i]    = (int32_t) pk.size();
        const int64_t b = ip[i + 1];
        if (ip[i] == b) pk.push_back(b);
        for (int64_t k = ip[i]; k < b;) {
            while (gi < gaps.size() && gaps[gi] <= k) ++gi;
            const int64_t cut = (gi < gaps.size() && gaps[gi] < b) ? gaps[gi] : b;
            pk.push_back(k);
            k = std::min(k + plen, cut);
        }
        if (pk.size() >= (size_t) INT32_MAX) return false;
    }
    row_piece[rows] = (int32_t) pk.size();
    pk.push_back(rows >= 0 ? ip[rows] : 0);
    return true;
}

// CSR-Adaptive segments of the row pointers ip[0..rows] (Idx: 32 or 64 bits):
// a row of more than `shrt` nonzeros is cut into `lng`-nonzero pieces (their
// segments in split: first, one past the last), shorter rows are packed, at
// most `shrt` nonzeros and `max_rows` rows a segment.  sk: first nonzero of
// each segment plus ip[rows]; si: its first row (bit 31: a piece of a long
// row) plus rows.  A packed segment ends at the last row that fits: found by
// bisection, not row by row (540 k rows of a field's voxel-major matrix: 0.4
// ms).  Returns false when the segments would not fit int32.
template<typename Idx>
static inline bool
cut_segments(const Idx* ip, int64_t rows, int64_t shrt, int64_t lng, int64_t max_rows, std::vector<int64_t>& sk,
             std::vector<uint32_t>& si, std::vector<int32_t>& split) {
    int64_t r = 0;
    while (r < rows) {
        const int64_t kb = (int64_t) ip[r], len = (int64_t) ip[r + 1] - kb;
        if (len > shrt) {
            split.push_back((int32_t) sk.size());
            for (int64_t off = 0; off < len; off += lng) {
                sk.push_back(kb + off);
                si.push_back((uint32_t) r | 0x80000000u);
            }
            split.push_back((int32_t) sk.size());
            ++r;
        } else {
            sk.push_back(kb);
            si.push_back((uint32_t) r);
            const Idx* e = ip + std::min(rows, r + max_rows) + 1;
            r = (std::upper_bound(ip + r + 1, e, (Idx) (kb + shrt)) - ip) - 1;
        }
        if (sk.size() >= (size_t) INT32_MAX) return false;
    }
    sk.push_back((int64_t) ip[rows]);
    si.push_back((uint32_t) rows);
    return true;
}

// A CSR handed in by a caller (rows x cols, row pointers ip[0..rows], column
// indices idx[0 .. ip[rows])): 0 when ip starts at 0 and does not decrease
// and every row's columns lie in [0, cols) and ascend strictly; else 1 (ip,
// *bad = the row), 2 (a column out of range) or 3 (columns not ascending),
// *bad = the entry.
static inline int
check_csr(int64_t rows, int64_t cols, const int64_t* ip, const int32_t* idx, int64_t* bad) {
    // the row pointers first: idx is read only up to ip[rows]
    if (ip[0] != 0) {
        *bad = 0;
        return 1;
    }
    for (int64_t i = 0; i < rows; ++i)
        if (ip[i + 1] < ip[i]) {
            *bad = i;
            return 1;
        }
    for (int64_t i = 0; i < rows; ++i) {
        for (int64_t k = ip[i]; k < ip[i + 1]; ++k) {
            if (idx[k] < 0 || (int64_t) idx[k] >= cols) {
                *bad = k;
                return 2;
            }
            if (k > ip[i] && idx[k] <= idx[k - 1]) {
                *bad = k;
                return 3;
            }
        }
    }
    return 0;
}

#endif
