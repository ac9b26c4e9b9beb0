// The cells that a node tile of the projection reads (k_p2m_tile): plain functions of the tile's
// first node, so the host can check them against the bounds of the start table.
//
// The cells of axis d run from -1 to n_d + 1 (stored index = cell + 1, cn_d = n_d + 3 of them); the
// table holds the first particle of each cell in x-fastest order and one end entry.  A tile's first
// node may lie far outside the grid: the block view reaches ncoarse nodes past it on every side.
#pragma once
#include <cstdint>

namespace vpmx {

constexpr int PT_X = 16, PT_Y = 4, PT_Z = 4;
constexpr int PC_X = PT_X + 3, PC_Y = PT_Y + 3, PC_Z = PT_Z + 3;
constexpr int PT_ROWS = PC_Y * PC_Z;

// Cell row r (0 .. PT_ROWS - 1) of the tile whose first node is (.., J0, K0), counted over the whole
// grid; -1 past its rows.
constexpr int64_t p2m_row(int J0, int K0, int r, int n1, int n2) {
    const int cj = J0 - 2 + r % PC_Y, ck = K0 - 2 + r / PC_Y;
    return cj >= -1 && cj <= n1 + 1 && ck >= -1 && ck <= n2 + 1 ? (cj + 1) + (int64_t)(n1 + 3) * (ck + 1) : -1;
}

// The start table's entry for cell column c (0 .. PC_X, the last one the row's end) of the tile whose
// first node is (I0, ..); `row` from p2m_row.  Columns past the grid take the row's first or end entry.
constexpr int64_t p2m_entry(int I0, int c, int64_t row, int n0) {
    const int cx = I0 - 2 + c, in = cx < -1 ? -1 : (cx > n0 + 2 ? n0 + 2 : cx);
    return row * (n0 + 3) + in + 1;
}

}  // namespace vpmx
