// Tables of a determinant list for its row build (see dets.hip).
#pragma once

#include <cstdint>

#include "kernels.h"

namespace cf {

// One connection of a string to another of the list's strings of its spin.
struct DetConn {
    uint32_t J;    // index of the other string
    uint8_t type;  // 0 itself, 1 single, 2 double excitation
    int8_t sign;   // singles
    uint8_t f, t;  // singles: orbital left and taken
    double x;      // singles: h_pq + sum_z (V_pzqz - V_pzzq); doubles: the element, this string first
    double xr;     // doubles: the element, the other string first
};

// The distinct strings of one spin, ascending, with their connections among
// themselves (ascending), and those of them that are no doubles.
struct DetStrings {
    uint64_t n = 0;
    DBuf<uint64_t> s;
    DBuf<double> d1;              // diag_one_string
    DBuf<int64_t> off, soff;      // n + 1 offsets into conn and sub
    DBuf<DetConn> conn, sub;
};

struct DetTables {
    uint64_t n = 0;
    DetStrings a, b;
    DBuf<uint32_t> ia, ib;  // string indices of each determinant, list order
    DBuf<uint32_t> pos;     // [a.n][b.n]: list index of the determinant, ~0: not in the list
};

// Builds the tables of a list of n distinct determinants from its sorted keys
// (up << 32 | down).  False, with nothing built, for a
// list that they do not suit: repeated determinants, more than 16,384 strings
// of a spin, or fewer than one determinant per 32 pairs of its strings (8 for
// lists of fewer than 4,096), which also bounds pos to 32 entries each.
bool make_det_tables(DetTables& T, uint64_t n, const str_t* up, const str_t* down, const uint64_t* skey, HamDev H,
                     hipStream_t stream);
// Count pass (r.rowcnt) or fill pass (r.rowptr, col, val, val32) of the rows.
// The fill writes a row's entries in the order of the sorted determinants:
// ascending columns for a list in (up, down) order.
void launch_det_rows_tab(const DetTables& T, const DetRowsArgs& r, bool fill, hipStream_t stream);

}  // namespace cf
