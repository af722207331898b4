// The automaton of csrc/bpe_automaton.hpp run over whole rows on the CPU, for tests/test_bpe_automaton.py.
#include "../../dnatok_amd/csrc/bpe_automaton.hpp"

extern "C" void *automaton_create(const int32_t *byte_to_sym, const int32_t *a, const int32_t *b, const int32_t *product,
                                  const uint8_t *in_effect, int32_t n_merges, int32_t n_symbols,
                                  int64_t max_states)
{
    dnatok::BpeAutomaton *fa = new dnatok::BpeAutomaton();
    if (dnatok::build_bpe_automaton(byte_to_sym, a, b, product, in_effect, n_merges, n_symbols, fa,
                                    max_states ? (size_t)max_states : dnatok::kAutoMaxStates)) return fa;
    delete fa;
    return nullptr;
}

extern "C" void automaton_destroy(void *h) { delete (dnatok::BpeAutomaton *)h; }

extern "C" int64_t automaton_max_states() { return (int64_t)dnatok::kAutoMaxStates; }

extern "C" int64_t automaton_states(const void *h) { return ((const dnatok::BpeAutomaton *)h)->n_states; }

// Tokens of a row into out; returns their number.
extern "C" int64_t automaton_encode(const void *h, const int32_t *byte_to_sym, const uint8_t *row, int64_t n, int32_t *out)
{
    const dnatok::BpeAutomaton &fa = *(const dnatok::BpeAutomaton *)h;
    std::vector<uint32_t> state(n + 1, 0);
    std::vector<uint8_t> foreign(n + 1, 0);
    uint32_t s = 0;
    for (int64_t i = 0; i < n; ++i) {
        const int c = (row[i] >> 1) & 3;
        if (((fa.letters >> (8 * c)) & 255u) == row[i]) {
            s = fa.next[4 * (size_t)s + c];
        } else {
            s = 0;                                   // behind a byte that is no letter a row starts anew
            foreign[i + 1] = 1;
        }
        state[i + 1] = s;
    }
    int64_t k = 0;
    for (int64_t p = n; p > 0;) {
        out[k++] = foreign[p] ? byte_to_sym[row[p - 1]] : (int32_t)fa.sym[state[p]];
        p -= foreign[p] ? 1 : fa.len[state[p]];
        if (p < 0) return -1;
    }
    std::reverse(out, out + k);
    return k;
}
