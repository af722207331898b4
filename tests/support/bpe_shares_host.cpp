// csrc/bpe_shares.hpp on the CPU, for tests/test_bpe_shares.py.
#include "../../dnatok_amd/csrc/bpe_shares.hpp"

// First row of every share into first[0 .. shares], and about which row it is looked for into guess[0 .. shares).
extern "C" void shares_deal(const int64_t *offsets, int32_t n_rows, int32_t shares, int32_t *first, int32_t *guess)
{
    const auto s = dnatok::RowShares<32>::of(offsets[0], offsets[n_rows], n_rows, shares, 1.0 / shares);
    int32_t row = 0;
    for (int32_t i = 0; i <= shares; ++i) {
        while (row < n_rows && s.cost_to(row, offsets[row]) < s.from(i)) ++row;
        first[i] = row;
        if (i < shares) guess[i] = i == 0 ? 0 : s.guess(i);
    }
}
