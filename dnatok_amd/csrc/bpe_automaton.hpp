// A BPE vocabulary as a finite automaton over the bytes of a row (host side: how it is built).
//
// Reading a row from left to right, call T(i) the last token of the encoding of the row's first i
// bytes.  Two facts about merge tables in which no rule's product is used by a lower-ranked rule:
//
//   * A sequence of tokens is the encoding of its string if and only if every two neighbours (s, t)
//     are: encode(s t) = [s, t].  (The first merge across a border of the sequence would happen in
//     the run on those two tokens alone as well: up to its rank both sides have the same history,
//     and of equal ranks the leftmost goes first.)  So whether t may follow s is a property of the
//     two tokens, called "t fits s" here.
//   * Hence T(i) is the one token t that ends at i and fits T(i - |t|), and the encoding of the
//     whole row is read off backwards: T(n), T(n - |T(n)|), ...
//
// What the T of later positions can depend on is, for every suffix of the text read so far that is a
// proper prefix of some token, which of those tokens fit the T in front of the suffix.  These sets
// are the states; they are few (8,972 for a vocabulary of 4,096 tokens over A C G T, 164,729 for one
// of 32,000), because a suffix is only remembered while a longer token can still complete it.
// Every state also names its T, so that a state sequence is all that is needed for the tokens.
//
// Whether t fits s: a rule (x, y) of rank r merges across the border if x, on the right edge of s,
// still stands at rank r (it is merged away as a right half at a higher rank), and y, on the left
// edge of t, does too; where both y's own merge and the rule have rank r (x x x: the rule (x, x)
// inside t), the pair across the border lies further left and goes first.
#pragma once

#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <string>
#include <vector>

namespace dnatok {

struct BpeAutomaton {
    uint32_t n_states = 0;             // state 0: nothing read yet (a row's start)
    std::vector<uint32_t> next;        // [4 * n_states] by letter code
    std::vector<uint8_t> len;          // [n_states] length of the state's last token
    std::vector<uint16_t> sym;         // [n_states] the last token itself
    uint32_t letters = 0;              // byte v of it: the byte whose code is v (a byte of another code where there is none)
};

// Limits beyond which a vocabulary has no automaton (its rows go to the merge engine): states, the
// suffixes they are made of, and the memory the construction takes for which token fits which.
// States: the most measured are 458,323 (60,000 tokens trained on text that is mostly repeats; 7.3 MB of
// transitions, beyond the 4 MB of an XCD's L2).  The states that text visits are far fewer, and the automaton is
// still ahead of the merges: 8,192 rows of 1 KB 187 -> 49 us, with repeats in a tenth of the bases 227 -> 117,
// 1,024 rows 66 -> 55, 32 of 100 kbp 164 -> 76.  (Only behind a copy of 512 MB are few rows with such repeats slower,
// 1,024 of 1 KB 65 -> 74 us.)  Creating such a table takes 0.4 s.
constexpr size_t kAutoMaxStates = 1u << 19;
constexpr size_t kAutoMaxItems = 1u << 22;
constexpr size_t kAutoMaxFitBytes = (size_t)256 << 20;
constexpr int kAutoMaxTokenLen = 255;

namespace automaton_detail {

constexpr int32_t kNever = 0x7FFFFFFF;

inline uint64_t mix(uint64_t h, uint64_t v)
{
    h = (h ^ v) * 0x9E3779B97F4A7C15ull;
    return h ^ (h >> 29);
}

// Open addressing map from 64-bit keys (no key is ~0) to 32-bit values.
class Map64 {
public:
    explicit Map64(size_t expect)
    {
        size_t n = 64;
        while (n < expect * 2) n <<= 1;
        key_.assign(n, ~0ull);
        val_.assign(n, 0);
    }
    uint32_t *find(uint64_t k)
    {
        const size_t m = key_.size() - 1;
        for (size_t i = mix(0, k) & m;; i = (i + 1) & m) {
            if (key_[i] == k) return &val_[i];
            if (key_[i] == ~0ull) return nullptr;
        }
    }
    void insert(uint64_t k, uint32_t v)
    {
        if ((n_ + 1) * 2 > key_.size()) grow();
        put(k, v);
        ++n_;
    }

private:
    void put(uint64_t k, uint32_t v)
    {
        const size_t m = key_.size() - 1;
        size_t i = mix(0, k) & m;
        while (key_[i] != ~0ull) i = (i + 1) & m;
        key_[i] = k; val_[i] = v;
    }
    void grow()
    {
        std::vector<uint64_t> k2(key_.size() * 2, ~0ull);
        std::vector<uint32_t> v2(key_.size() * 2, 0);
        k2.swap(key_); v2.swap(val_);
        for (size_t i = 0; i < k2.size(); ++i)
            if (k2[i] != ~0ull) put(k2[i], v2[i]);
    }
    std::vector<uint64_t> key_;
    std::vector<uint32_t> val_;
    size_t n_ = 0;
};

}  // namespace automaton_detail

// Builds the automaton of a merge table whose rules are in effect in rank order (`in_effect[i]` = 0:
// rule i was replaced by a later entry of the same pair) and in which no rule's product is used by a
// lower-ranked rule.  False: this table has none (more than four bytes with rules, bytes whose bits 1
// and 2 do not tell them apart, tokens of more than 255 bytes, symbols that stand for more than one
// string, or more states than the limits).
inline bool build_bpe_automaton(const int32_t *byte_to_sym, const int32_t *pair_a, const int32_t *pair_b,
                                const int32_t *product, const uint8_t *in_effect, int32_t n_merges, int32_t n_symbols,
                                BpeAutomaton *out, size_t max_states = kAutoMaxStates)
{
    using namespace automaton_detail;
    if (n_merges <= 0) return false;

    // the letters: bytes whose symbols take part in rules
    std::vector<int32_t> byte_of(n_symbols, -1);                   // -2: more than one byte
    for (int v = 0; v < 256; ++v) byte_of[byte_to_sym[v]] = byte_of[byte_to_sym[v]] == -1 ? v : -2;
    int32_t letter_sym[4] = {-1, -1, -1, -1};
    std::vector<int8_t> code_of(n_symbols, -1);
    for (int32_t r = 0; r < n_merges; ++r) {
        if (!in_effect[r]) continue;
        if (byte_of[product[r]] != -1) return false;               // a rule that makes a single byte's symbol
        for (int32_t s : {pair_a[r], pair_b[r]}) {
            if (byte_of[s] == -1 || code_of[s] >= 0) continue;
            if (byte_of[s] == -2) return false;
            const int c = (byte_of[s] >> 1) & 3;
            if (letter_sym[c] >= 0) return false;
            letter_sym[c] = s;
            code_of[s] = (int8_t)c;
        }
    }
    uint32_t letters = 0;
    for (int c = 0; c < 4; ++c) {
        const int v = letter_sym[c] >= 0 ? byte_of[letter_sym[c]] : ((c ^ 1) << 1);     // (no letter: a byte whose code differs)
        letters |= (uint32_t)v << (8 * c);
    }

    // how each token comes about: its last rule, and through it both of its edges
    Map64 rank_of((size_t)n_merges);
    for (int32_t r = 0; r < n_merges; ++r)
        if (in_effect[r]) rank_of.insert((uint64_t)pair_a[r] << 32 | (uint32_t)pair_b[r], (uint32_t)r);
    std::vector<int32_t> left(n_symbols, -1), right(n_symbols, -1), made(n_symbols, -1);
    std::vector<std::string> text(n_symbols);
    for (int c = 0; c < 4; ++c)
        if (letter_sym[c] >= 0) text[letter_sym[c]] = std::string(1, (char)c);
    // does a rule below rank `limit` merge across the border of s t?
    auto crossed = [&](int32_t s, int32_t t, int32_t limit) {
        int32_t gone_x = kNever;
        for (int32_t x = s;;) {
            int32_t gone_y = kNever;
            for (int32_t y = t;;) {
                const uint32_t *r = rank_of.find((uint64_t)x << 32 | (uint32_t)y);
                if (r && (int32_t)*r < limit && (int32_t)*r < gone_x && (int32_t)*r <= gone_y) return true;
                if (made[y] < 0) break;
                gone_y = made[y];
                y = left[y];
            }
            if (made[x] < 0) break;
            gone_x = made[x];
            x = right[x];
        }
        return false;
    };
    for (int32_t r = 0; r < n_merges; ++r) {
        if (!in_effect[r]) continue;
        const int32_t a = pair_a[r], b = pair_b[r], p = product[r];
        if (text[a].empty() || text[b].empty()) continue;          // a side that no text ever becomes
        if (crossed(a, b, r)) continue;                            // a b never meet as neighbours
        if (made[p] >= 0) {
            if (text[p] != text[a] + text[b]) return false;
            continue;
        }
        if (text[a].size() + text[b].size() > (size_t)kAutoMaxTokenLen) return false;
        left[p] = a; right[p] = b; made[p] = r;
        text[p] = text[a] + text[b];
    }

    // the tokens in the order of their texts: those with a common prefix are neighbours
    std::vector<int32_t> order;
    for (int32_t s = 0; s < n_symbols; ++s)
        if (!text[s].empty()) order.push_back(s);
    std::sort(order.begin(), order.end(), [&](int32_t p, int32_t q) { return text[p] < text[q]; });
    const int32_t n_tok = (int32_t)order.size();
    std::vector<int32_t> place(n_symbols, -1);
    for (int32_t i = 0; i < n_tok; ++i) place[order[i]] = i;
    // the tree of their prefixes; [lo, hi): the places of the tokens that go on beyond the node
    struct Node {
        int32_t child[4];
        int32_t token, lo, hi;
    };
    std::vector<Node> tree(1, Node{{-1, -1, -1, -1}, -1, 0, n_tok});
    for (int32_t i = 0; i < n_tok; ++i) {
        int32_t at = 0;
        for (char ch : text[order[i]]) {
            int32_t &to = tree[at].child[(int)ch];
            if (to < 0) {
                const int32_t fresh = (int32_t)tree.size();
                to = fresh;                                        // (before push_back moves the node)
                tree.push_back(Node{{-1, -1, -1, -1}, -1, i, i});
                at = fresh;
            } else {
                at = to;
            }
            tree[at].hi = i + 1;
        }
        if (tree[at].token >= 0) return false;                     // two symbols of one text
        tree[at].token = order[i];
        tree[at].lo = i + 1;                                       // (the token itself comes first of its subtree)
    }

    // Which tokens do not fit a token s, as bits by place.  It depends on the rules that s's right
    // edge can still take part in, so tokens with the same such rules share a row of bits.
    std::vector<std::vector<int32_t>> rules_of(n_symbols);         // rules by left side, in rank order
    for (int32_t r = 0; r < n_merges; ++r)
        if (in_effect[r]) rules_of[pair_a[r]].push_back(r);
    std::vector<std::vector<std::pair<int32_t, int32_t>>> begins(n_symbols);     // y -> {rank at which it goes, place of the token}
    for (int32_t i = 0; i < n_tok; ++i) {
        int32_t gone = kNever;
        for (int32_t y = order[i];; y = left[y]) {
            begins[y].push_back({gone, i});
            if (made[y] < 0) break;
            gone = made[y];
        }
    }
    struct Edge { int32_t x, n_rules, row; };
    std::vector<Edge> edges;
    std::vector<int32_t> row_of(n_symbols, -1);
    int32_t n_rows = 1;                                            // row 0: nothing in front, everything fits
    {
        Map64 seen((size_t)n_tok);
        std::vector<std::vector<int32_t>> key_of_row(1);
        std::vector<int32_t> chain(1, -1), key;                    // rows whose keys share a hash
        for (int32_t i = 0; i < n_tok; ++i) {
            key.clear();
            int32_t gone = kNever;
            for (int32_t x = order[i];; x = right[x]) {
                const std::vector<int32_t> &ru = rules_of[x];
                const int32_t k = (int32_t)(std::lower_bound(ru.begin(), ru.end(), gone) - ru.begin());
                if (k) { key.push_back(x); key.push_back(k); }
                if (made[x] < 0) break;
                gone = made[x];
            }
            uint64_t h = 1;
            for (int32_t v : key) h = mix(h, (uint32_t)v);
            h >>= 1;
            uint32_t *head = seen.find(h);
            int32_t row = head ? (int32_t)*head : -1;
            while (row >= 0 && key_of_row[row] != key) row = chain[row];
            if (row < 0) {
                row = n_rows++;
                key_of_row.push_back(key);
                chain.push_back(head ? (int32_t)*head : -1);
                if (head) *head = (uint32_t)row; else seen.insert(h, (uint32_t)row);
                for (size_t q = 0; q < key.size(); q += 2) edges.push_back(Edge{key[q], key[q + 1], row});
            }
            row_of[order[i]] = row;
        }
    }
    const size_t words = ((size_t)n_tok + 63) / 64;
    if ((size_t)n_rows * words * 8 > kAutoMaxFitBytes) return false;
    std::vector<uint64_t> unfit((size_t)n_rows * words, 0);
    std::sort(edges.begin(), edges.end(), [](const Edge &p, const Edge &q) {
        return p.x != q.x ? p.x < q.x : (p.n_rules != q.n_rules ? p.n_rules < q.n_rules : p.row < q.row);
    });
    {
        std::vector<uint64_t> bits(words);
        size_t lo_w = words, hi_w = 0;                             // the words of `bits` in use
        for (size_t e = 0; e < edges.size();) {
            const int32_t x = edges[e].x;
            for (size_t w = lo_w; w < hi_w; ++w) bits[w] = 0;
            lo_w = words; hi_w = 0;
            int32_t k = 0;
            for (; e < edges.size() && edges[e].x == x; ++e) {
                for (; k < edges[e].n_rules; ++k) {
                    const int32_t r = rules_of[x][k];
                    for (const auto &b : begins[pair_b[r]])
                        if (b.first >= r) {
                            const size_t w = (size_t)b.second >> 6;
                            bits[w] |= 1ull << (b.second & 63);
                            lo_w = std::min(lo_w, w);
                            hi_w = std::max(hi_w, w + 1);
                        }
                }
                uint64_t *row = &unfit[(size_t)edges[e].row * words];
                for (size_t w = lo_w; w < hi_w; ++w) row[w] |= bits[w];
            }
        }
    }
    auto fits = [&](int32_t row, int32_t at) { return !(unfit[(size_t)row * words + ((size_t)at >> 6)] >> (at & 63) & 1); };

    // A suffix in a state: a node of the tree and the tokens beyond it that fit what is in front.
    // Equal nodes with equal sets are one item; 0: no token is left.  What a letter makes of an item
    // (the item of the longer suffix, and the token that is complete with it, if it fits) is found once.
    struct Item { int32_t row, node; };
    struct Step { uint32_t item; int32_t token; };
    std::vector<Item> items(1, Item{0, 0});
    std::vector<Step> steps(4, Step{0, -1});                       // [4 * item + letter]
    std::vector<uint32_t> item_chain(1, 0);
    Map64 item_by_set(1 << 15);
    auto word_of = [&](int32_t row, int32_t lo, int32_t hi, int32_t w) {
        uint64_t m = ~unfit[(size_t)row * words + (size_t)w];
        if (w == lo >> 6) m &= ~0ull << (lo & 63);
        if (w == (hi - 1) >> 6 && (hi & 63)) m &= (1ull << (hi & 63)) - 1;
        return m;
    };
    auto item_of = [&](int32_t row, int32_t node) -> uint32_t {
        const int32_t lo = tree[node].lo, hi = tree[node].hi;
        if (lo >= hi) return 0;
        uint64_t h = (uint64_t)node + 1;
        bool any = false;
        for (int32_t w = lo >> 6; w <= (hi - 1) >> 6; ++w) {
            const uint64_t m = word_of(row, lo, hi, w);
            any |= m != 0;
            h = mix(h, m);
        }
        if (!any) return 0;
        h >>= 1;
        uint32_t *head = item_by_set.find(h);
        for (uint32_t id = head ? *head : 0; id; id = item_chain[id]) {
            if (items[id].node != node) continue;
            bool same = items[id].row == row;
            for (int32_t w = lo >> 6; !same; ++w) {
                if (word_of(row, lo, hi, w) != word_of(items[id].row, lo, hi, w)) break;
                same = w == (hi - 1) >> 6;
            }
            if (same) return id;
        }
        const uint32_t id = (uint32_t)items.size();
        items.push_back(Item{row, node});
        item_chain.push_back(head ? *head : 0);
        if (head) *head = id; else item_by_set.insert(h, id);
        return id;
    };
    auto step_items = [&] {
        for (uint32_t id = (uint32_t)(steps.size() / 4); id < items.size() && items.size() <= kAutoMaxItems; ++id)
            for (int c = 0; c < 4; ++c) {
                const Item it = items[id];
                const int32_t node = tree[it.node].child[c];
                Step st{0, -1};
                if (node >= 0) {
                    const int32_t token = tree[node].token;
                    if (token >= 0 && fits(it.row, place[token])) st.token = token;
                    st.item = item_of(it.row, node);
                }
                steps.push_back(st);
            }
    };
    std::vector<uint32_t> behind(n_rows);                          // the item of "nothing yet" behind a token, by its row
    for (int32_t r = 0; r < n_rows; ++r) behind[r] = item_of(r, 0);
    step_items();
    if (items.size() > kAutoMaxItems) return false;

    // The states reachable from a row's start.  A state is its items, longest suffix first, and its
    // last token; state s's lie in pool[first[s] .. first[s + 1]).
    std::vector<uint32_t> pool, state_chain, cand;
    std::vector<size_t> first(1, 0);
    Map64 state_by_key(1 << 15);
    out->next.clear(); out->len.clear(); out->sym.clear();
    auto state_of = [&](const std::vector<uint32_t> &key) -> uint32_t {
        uint64_t h = key.size();
        for (uint32_t v : key) h = mix(h, v);
        h >>= 1;
        uint32_t *head = state_by_key.find(h);
        for (uint32_t s = head ? *head : ~0u; s != ~0u; s = state_chain[s])
            if (first[s + 1] - first[s] == key.size() &&
                memcmp(&pool[first[s]], key.data(), key.size() * sizeof(uint32_t)) == 0) return s;
        const uint32_t s = (uint32_t)state_chain.size();
        pool.insert(pool.end(), key.begin(), key.end());
        first.push_back(pool.size());
        state_chain.push_back(head ? *head : ~0u);
        if (head) *head = s; else state_by_key.insert(h, s);
        return s;
    };
    cand.assign({behind[0], ~0u});
    (void)state_of(cand);
    out->len.push_back(1);
    out->sym.push_back(0);
    for (uint32_t s = 0; s < state_chain.size(); ++s) {
        if (state_chain.size() > max_states) return false;
        for (int c = 0; c < 4; ++c) {
            if (letter_sym[c] < 0) { out->next.push_back(0); continue; }
            int32_t last = -1;
            cand.clear();
            for (size_t i = first[s]; i + 1 < first[s + 1]; ++i) {
                const Step st = steps[4 * (size_t)pool[i] + c];
                if (last < 0) last = st.token;
                if (st.item) cand.push_back(st.item);
            }
            if (last < 0) return false;
            if (const uint32_t id = behind[row_of[last]]) cand.push_back(id);
            cand.push_back((uint32_t)last);
            const uint32_t to = state_of(cand);
            if (to == out->len.size()) {
                out->len.push_back((uint8_t)text[last].size());
                out->sym.push_back((uint16_t)last);
            }
            out->next.push_back(to);
        }
    }
    if (state_chain.size() > max_states) return false;
    out->n_states = (uint32_t)state_chain.size();
    out->letters = letters;
    return true;
}

}  // namespace dnatok
