// How the rows of a large batch are dealt out to the waves of the BPE automaton: in shares of about one cost, by
// where the rows lie and without a pass over them.  Plain C++ for the device and for the host (its test).
#pragma once

#include <stdint.h>

#ifdef __HIPCC__
#define DNATOK_SHARES_FN __host__ __device__ __forceinline__
#else
#define DNATOK_SHARES_FN inline
#endif

namespace dnatok {

// A row costs its bytes and a region of kRegion bytes: never less than the lanes it takes (a region each, the
// last one begun, and one for an empty row).  What the rows in front of row r cost is the bytes in front of it and r
// regions, so a row's place in the batch's cost needs nothing but the row's own offset, and it grows with every
// row: a share holds at most each / kRegion + 1 rows.  (With the bytes alone as the cost, a run of empty rows was one
// share: see launch_auto_as.)
template <int kRegion>
struct RowShares {
    int64_t base;                // where the batch's first row starts
    int64_t each;                // cost of a share
    int32_t shares;
    float rows_per_cost;

    // `end`: where the last row ends; inv_shares: 1.0 / shares
    static DNATOK_SHARES_FN RowShares of(int64_t begin, int64_t end, int32_t n_rows, int32_t shares, double inv_shares)
    {
        const int64_t cost = end - begin + (int64_t)kRegion * n_rows;
        return RowShares{begin, (int64_t)((double)cost * inv_shares) + 1, shares, (float)n_rows / (float)cost};
    }
    // what the rows in front of `row` cost, which starts at `offset`
    DNATOK_SHARES_FN int64_t cost_to(int64_t row, int64_t offset) const { return offset - base + kRegion * row; }
    // a share is the rows with cost_to() in [from(i), from(i + 1)); the last one takes what rounding leaves
    DNATOK_SHARES_FN int64_t from(int64_t i) const { return i <= 0 ? INT64_MIN : i >= shares ? INT64_MAX : i * each; }
    // about which row share i > 0 begins at
    DNATOK_SHARES_FN int32_t guess(int64_t i) const { return (int32_t)((float)(i * each) * rows_per_cost); }
};

}  // namespace dnatok
