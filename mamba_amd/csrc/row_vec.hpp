// Which elements of a row the causal conv's kernels read for the VW
// consecutive ones at i (a multiple of VW, from -VW on).  Plain constexpr, so
// that the kernels and a host program share the rule.
#pragma once
#include <cstdint>

namespace ss {

// whether element i exists in a row of n
constexpr bool row_in(int64_t i, int64_t n) { return i >= 0 && i < n; }
// i, or the nearest element that exists
constexpr int64_t row_elem(int64_t i, int64_t n) { return i < 0 ? 0 : (i >= n ? n - 1 : i); }
// Rows of whole vectors, rows that end inside one, and rows shorter than one
// (fixed per launch: a test of the length beside each load cost the ragged
// rows 1-3 % of a forward + backward at batch 8 x 1536 x 2047 bf16).
enum class Rows { kWhole, kRagged, kShort };
constexpr Rows rows_of(int64_t n, int vw) { return n < vw ? Rows::kShort : n % vw ? Rows::kRagged : Rows::kWhole; }
// One vector load, at row_vec_at, does for the vector at i: it lies wholly
// inside the row, or wholly outside and the row's first vector is read in its
// place.  Not where it straddles the row's end, and nowhere in a short row:
// those are read element by element, at row_elem.
constexpr int64_t row_vec_at(int64_t i, int64_t n) { return row_in(i, n) ? i : 0; }
constexpr bool row_vec_ok(Rows rows, int64_t i, int64_t n, int vw) {
    return rows == Rows::kWhole || (rows == Rows::kRagged && !(row_in(i, n) && i + vw > n));
}

}  // namespace ss
