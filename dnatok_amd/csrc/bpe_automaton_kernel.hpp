// The BPE automaton on the device: rows and chunks of at most 64 * P bytes, a few lanes per row.
// Included by bpe_encode.hip (bpe_automaton.hpp has what the automaton is and why it gives the
// encoding).
//
// A row is cut into regions of P bytes, one per lane; a wave holds as many rows as fit its lanes.
//   forward    Every lane runs the automaton over its region from the row-start state and keeps the
//              state behind every byte in LDS.  A lane then goes on into the next lane's region,
//              replacing what it finds there, until it meets the state that is there already: from
//              then on both runs are the same, so the states are those of the run from the row's
//              start.  (Lanes that reach the end of that region go on into the one after it.)  Two
//              runs meet within a few tokens of their first common border; inside a tandem repeat
//              they may not, and the lanes walk on to its end.
//   backward   The tokens are read off from the row's end: the state behind byte p - 1 names the token
//              that ends at p.  Every lane does this for its region from the region's own end first,
//              noting the token starts as bits; then it is told where the token that reaches into its
//              region really starts (by the lane to its right), walks from there until it meets a start
//              it has, and passes its own border on if that moved.
//   output     The lanes' counts give every token its number; tokens go through LDS into place and out
//              of it in whole vectors (ids, padding and mask), or, for a chunk of a long row, to the
//              positions they start at, as the seam and gather kernels expect them.
//
// What bounds it: the forward walk is a chain of dependent reads, one per byte and lane, so the
// transition table has to be near.  Narrow form: 16-bit transitions and the token lengths in LDS,
// staged once per workgroup, one workgroup of up to sixteen waves per CU (8,972 states: 81 KB, and 5 KB
// per wave for states and tokens).  Wide form: 32-bit entries {state, token length} in global memory
// (L2: 164,729 states are 2.6 MB).  (With the transitions of the first 4,992 states, where every second
// step is, in LDS as well, the walk over the own region went from 10.7 to 7.8 us, staging them took the 3 us
// back, and the walk into the next region, a few lanes inside tandem repeats, stayed at 16 us.)
//
// Every phase is a chain of dependent reads, so what a launch takes is the number of waves in flight.
// Sixteen share the table instead of eight since a wave's tokens leave through a window of one per four
// bytes (more than that are written lane by lane) and a chunk's go where the states were: 16,384 rows of
// 1 KB 54.7 -> 29.2 us, 100,000 reads 123 -> 57 us.  (That includes the walk into the next region four bytes
// at a time, comparing the last of the four, and the padded rows of a wave written as one run of cells.)
//
// Per call, the merge engine -> the automaton: 1,024 rows of 1 KB 29.4 -> 11.7 us, 16,384 of them 236.5 ->
// 26.9 us, 100,000 reads of 100 - 300 bp (int64 rows) 349 -> 49.5 us, 4,096 ragged reads of 12 Mbp 253.5 ->
// 79 us (all with the vocabulary of 4,096), 32 rows of 100 kbp (32,000) 143.8 -> 59.6 us.
//
// Beside the chains of dependent reads vector issue is what a full chip runs out of (three fifths of the time), so the
// steps of the chains are as few instructions as they can be: an entry and a code are the next entry's address in one
// (32-bit entries on their way, the table at the start of LDS), a word's codes are gathered by one dot product, which
// bytes are no letters is looked at where there are any, and the walk backwards notes the ends of tokens: 16,384 rows of
// 1 KB 1,144 -> 933 vector instructions per step.
#pragma once

namespace dnatok {

struct AutoArgs {
    const void *next;            // narrow: uint16 [4 * (n_states + 1)], entry = 4 * state; wide: uint32, entry = 4 * state << 8 | length
    const uint8_t *len;          // [n_states + 1] (narrow)
    const uint16_t *sym;         // [n_states + 1 + 256] token of a state; behind the states: symbol of a byte
    const int32_t *id;           // the same through the table's out_remap
    uint32_t other;              // the state behind a byte that is no letter; its successors are the row start's
    uint32_t letters;            // the letters by code (bits 1 and 2 of the byte)
    int32_t rows;                // (whole rows) rows of an item, at most 64
    int32_t n_groups;            // (whole rows) items (chunks: the work list says)
    int32_t window;              // tokens a wave has room for on their way out
    int32_t list_here;           // (chunks) the kernel makes the work list itself: at most kAutoListRows rows
    int32_t entries_here;        // (chunks) the list says where a row's chunks begin, their entries are written here (auto_entries_here)
    int32_t *zero;               // (chunks) a word to be cleared for the kernels behind this one, or null
    int64_t total;               // bytes of the batch
};

// Waves of a workgroup, which has a CU to itself: as many as the LDS holds, at most sixteen (four per SIMD).
constexpr int kAutoMaxWaves = 16;
constexpr uint32_t kAutoNarrowStates = 10400;    // the most the narrow form has LDS for, beside the waves' share
constexpr size_t kAutoLdsBytes = 163840;         // a CU's
constexpr size_t kAutoLdsAside = 1152;           // of it, for what is neither table nor a wave's (the longest rows, or the characters' ids)

typedef uint32_t auto_u32_a1 __attribute__((aligned(1), may_alias));
typedef uint32_t auto_u32x4_a1 __attribute__((ext_vector_type(4), aligned(1), may_alias));
typedef int32_t auto_i32x4 __attribute__((ext_vector_type(4)));

template <bool WIDE, int P>
struct AutoLds {
    typedef typename std::conditional<WIDE, uint32_t, uint16_t>::type Entry;
    static constexpr size_t state_bytes = 64 * P * sizeof(Entry);
    static constexpr int least_window = 16 * P;                            // a token per four bytes
    static size_t table_bytes(uint32_t n_states)
    {
        return WIDE ? 0 : ((((size_t)n_states + 1) * 8 + 15) & ~(size_t)15) + ((((size_t)n_states + 1) + 15) & ~(size_t)15);
    }
    static int waves(uint32_t n_states)
    {
        const size_t w = (kAutoLdsBytes - kAutoLdsAside - table_bytes(n_states)) / (state_bytes + least_window * sizeof(Entry));
        return w > (size_t)kAutoMaxWaves ? kAutoMaxWaves : (int)w;
    }
    static int window(uint32_t n_states)
    {
        const size_t w = ((kAutoLdsBytes - kAutoLdsAside - table_bytes(n_states)) / waves(n_states) - state_bytes) / sizeof(Entry) & ~(size_t)7;
        return w > (size_t)(64 * P) ? 64 * P : (int)w;
    }
    static size_t bytes(uint32_t n_states)
    {
        return table_bytes(n_states) + waves(n_states) * (state_bytes + window(n_states) * sizeof(Entry)) + kAutoLdsAside;
    }
};

// From this many bytes on, walked into the regions to the right, a lane looks for a repeat: twice what a walk takes
// in other text, and behind it lies the longest period of the states in the common repeats (80 bytes).  (From 96
// bytes on, rows with short repeats in them, 10 % of their bases, were 3 % slower, 28.8 -> 29.6 us for 1,024 of 1 KB
// with the vocabulary of 32,000; from 128 on they are 3 % faster, 27.8 us.)
constexpr int kRepeatsFrom = 128;

// Up to this many rows a wave finds its item among the rows itself (their lengths are one load per 64
// rows, beside each other) instead of in a list that a launch in front has made: 5 us per call, as long
// as anything that a batch of a few rows waits for.
constexpr int kAutoListRows = 256;

// Up to this many rows a wave finds its chunk's row among the rows' first chunks (two trips, where the list's entry is
// one) and writes the entry for the kernels behind; with more, bpe_expand_kernel has written the entries.  A launch less,
// or the work list's kernel without that part: 2,000 rows of 5 kbp 53.5 -> 50.2 us, 900 of 20 kbp 77.2 -> 72.8, 2,500 of 4 kbp
// 59.2 -> 53.6, 4,096 ragged reads of 12 Mbp 54.4 -> 53.9 (one call on its own).  The search is made for every chunk and its
// trips grow with the rows, so a batch of many rows stays with the entries where a wave has a third chunk: 3,000 rows of
// 5 kbp 65.8 us, searched for 67.0, 4,096 of them 75.7 / 76.7, 4,097 78.5 / 83.2, 16,384 241.7 / 253.2, 50,000 ragged 425.8 / 444.9.
constexpr int kAutoEntryRows = 4096;
constexpr int kAutoEntryManyRows = 2048;                   // from here on
constexpr int kAutoEntryChunks = 7168;                     // as many chunks by the batch's bytes (about 8,192 with what the rows' ends leave), two to a wave
inline bool auto_entries_here(int64_t n_rows, int64_t total, int64_t core)
{
    return n_rows > kAutoListRows && n_rows <= kAutoEntryRows && (n_rows <= kAutoEntryManyRows || total <= kAutoEntryChunks * core);
}

constexpr uint32_t kXcds = 8;                    // (workgroups go to them in turn)

// 16 bits at an address of LDS (a kernel's dynamic array begins at 0 where it has no other)
__device__ __forceinline__ uint32_t lds_u16(uint32_t at)
{
    uint32_t v = *reinterpret_cast<const __attribute__((address_space(3))) uint16_t *>(at);
    asm("" : "+v"(v));                                  // (else the compiler forgets that the read has cleared the upper half)
    return v;
}

// Between two phases of a wave's work on its LDS: what a lane wrote before is what the others read after.
__device__ __forceinline__ void wave_phase()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Codes of the 16 bytes of w (two bits each, the first byte lowest: a word's four by one dot product with 1, 4, 16,
// 64); differs: has a bit wherever a byte is no letter.
__device__ __forceinline__ uint32_t letter_codes16(const auto_u32x4_a1 w, uint32_t letters, uint32_t &differs)
{
    uint32_t codes = 0;
    differs = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const uint32_t sel = (w[q] >> 1) & 0x03030303u;
        differs |= __builtin_amdgcn_perm(letters, letters, sel) ^ w[q];
        codes |= __builtin_amdgcn_udot4(sel, 0x40100401u, 0u, false) << (8 * q);
    }
    return codes;
}

// Which of the 16 bytes of w are no letters.
__device__ __forceinline__ uint32_t foreign16(const auto_u32x4_a1 w, uint32_t letters)
{
    uint32_t bad = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const uint32_t d = __builtin_amdgcn_perm(letters, letters, (w[q] >> 1) & 0x03030303u) ^ w[q];
        // the high bit of every byte that differs, then four bits together
        const uint32_t hi = ((d & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | d;
        bad |= __builtin_amdgcn_udot4((hi >> 7) & 0x01010101u, 0x08040201u, 0u, false) << (4 * q);
    }
    return bad;
}

// One id, in the padded output's own integer width.
__device__ __forceinline__ void auto_put(void *ids, int elem, int64_t at, int32_t v)
{
    if (elem == 4) reinterpret_cast<int32_t *>(ids)[at] = v;
    else if (elem == 8) reinterpret_cast<int64_t *>(ids)[at] = (int64_t)v;
    else if (elem == 2) reinterpret_cast<int16_t *>(ids)[at] = (int16_t)v;
    else reinterpret_cast<uint8_t *>(ids)[at] = (uint8_t)v;
}

// `rows` rows of the padded output, whose tokens lie in `staged`: lane first + r knows the number of the
// r-th of them, and that its n_tok tokens lie from `base` on.  The rows are taken as one run of cells,
// four to a lane (they start on such a boundary).
template <int ELEM, typename Entry>
__device__ __forceinline__ void auto_put_rows(const BpeArgs &a, const int32_t *id, const Entry *staged, int base, int n_tok,
                                              int first, int rows, int32_t row_id, int lane)
{
    const int stride = (int)a.pad_stride, quads = stride >> 2;
    const int64_t n_steps = ((int64_t)rows * quads + 63) >> 6;
    int r = 0, c = lane;
    for (int64_t step = 0; step < n_steps; ++step, c += 64) {
        while (c >= quads && r < rows) { c -= quads; ++r; }
        const int from = first + (r < rows ? r : 0);
        const int n = __shfl(n_tok, from), b = __shfl(base, from);
        const int64_t row = __shfl(row_id, from);
        if (r < rows) {
            const int kept = n < stride ? n : stride;
            const int shift = a.pad_left ? stride - kept : 0;
            const Entry *const st = staged + b;
            int32_t v[4];
            uint32_t live = 0;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int t = 4 * c + q - shift;
                const bool token = t >= 0 && t < kept;
                v[q] = a.pad_id;
                if (token) v[q] = id[st[t]];
                live |= (token ? 1u : 0u) << (8 * q);
            }
            if (a.pad_remap) {
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (live >> (8 * q) & 1u) v[q] = a.pad_remap[v[q]];
            }
            const int64_t at = row * stride + 4 * c;
            if (ELEM == 4) {
                *reinterpret_cast<auto_i32x4 *>(reinterpret_cast<int32_t *>(a.pad_ids) + at) = auto_i32x4{v[0], v[1], v[2], v[3]};
            } else if (ELEM == 8) {
                auto_i32x4 *const o = reinterpret_cast<auto_i32x4 *>(reinterpret_cast<int64_t *>(a.pad_ids) + at);
                o[0] = auto_i32x4{v[0], v[0] >> 31, v[1], v[1] >> 31};
                o[1] = auto_i32x4{v[2], v[2] >> 31, v[3], v[3] >> 31};
            } else if (ELEM == 2) {
                *reinterpret_cast<uint2 *>(reinterpret_cast<int16_t *>(a.pad_ids) + at) =
                    uint2{((uint32_t)v[0] & 0xFFFFu) | ((uint32_t)v[1] << 16), ((uint32_t)v[2] & 0xFFFFu) | ((uint32_t)v[3] << 16)};
            } else {
                *reinterpret_cast<uint32_t *>(reinterpret_cast<uint8_t *>(a.pad_ids) + at) =
                    ((uint32_t)v[0] & 0xFFu) | (((uint32_t)v[1] & 0xFFu) << 8) | (((uint32_t)v[2] & 0xFFu) << 16) | ((uint32_t)v[3] << 24);
            }
            if (a.pad_mask) *reinterpret_cast<uint32_t *>(a.pad_mask + at) = live;
        }
    }
}

// Lanes that have gone on (`going`, with state e) through the regions up to lane + ahead - 1 without meeting
// the state that was there: inside a tandem repeat the run from the row's start and a run that began inside
// may differ in phase for as long as it lasts.  But where a run's state is the one it had d bytes before, and
// the bytes from here on are those d bytes before them, its next states are those of d bytes before as well.
// So the walkers' last states are compared with the states of their own run behind them, all distances at once,
// the regions ahead whose bytes repeat at such a distance are counted, and their states copied by their own
// lanes; the walk goes on behind them, as that of the lane `ahead` regions before.  A row of 2,048 bases that is
// one repeat takes at most 136 steps of the automaton in a row instead of 2,048: 64 rows of 2,000 bases of A, AC, AAT,
// AAAT or AACCG with the vocabulary of 32,000 155 - 171 -> 23 - 26 us (the merge engine: 65 - 105), of AAT with that
// of 4,096 117 -> 18.5 us (36).  Rows that never come here are 0.2 - 1.7 % slower for the code in their way (16,384
// rows of 1 KB 28.5 -> 29.0 us); as a function of its own, or with a second copy of the walk for it, 2 - 5 %.
// A walker's run behind it is only its own where no other walker of the row has come by since: not those
// with a walker less than `ahead` lanes to their left.
template <int P, typename Entry>
__device__ __forceinline__ void copy_repeats(Entry *state, const uint32_t (&codes)[P / 16], uint32_t flags, bool any_foreign, int cnt,
                                             int cnt_ahead, int lane, int lane0, int lane_end, int ahead, uint32_t &e, bool &going)
{
    constexpr int kTries = 4, kLongest = 256;              // walkers per call, and distances of one of them; the longest distance
    const int behind = ahead * P < kLongest ? ahead * P : kLongest;
    const uint64_t mine = P == 32 ? (uint64_t)codes[P / 16 - 1] << 32 | codes[0] : codes[0];
    int done = -1;
#pragma unroll 1
    for (int tries = 0; tries < kTries; ++tries) {
        const uint64_t left = __ballot(going) & ((1ull << lane) - 1ull);
        const int nearest = left ? 63 - __builtin_clzll(left) : -1;
        const uint64_t eligible = __ballot(going && lane > done && (nearest < lane0 || lane - nearest >= ahead));
        if (!eligible) break;
        const int walker = __builtin_ctzll(eligible);
        const int first = walker + ahead;                  // the region it is about to enter
        const int row_end = __builtin_amdgcn_readlane(lane_end, walker);
        const uint32_t now = (uint32_t)__builtin_amdgcn_readlane((int)e, walker);
        int k = 0, d = 0, looked = 0;
#pragma unroll 1
        for (int d0 = 1; k == 0 && looked < kTries && d0 < behind; d0 += 64) {
            const int back = d0 + lane;
            bool same = false;
            if (back < behind) {
                const int pos = first * P - 1 - back;
                same = state[(pos & (P - 1)) * 64 + pos / P] == now;
            }
            uint64_t at = __ballot(same);
            while (at && k == 0 && looked < kTries) {
                d = d0 + __builtin_ctzll(at);
                at &= at - 1;
                ++looked;
                // the region's bytes against those d before them
                const int regions = (d + P - 1) / P, o = regions * P - d;
                const int from = lane - regions;
                uint64_t lo = (uint32_t)__shfl((int)codes[0], from & 63), hi = (uint32_t)__shfl((int)codes[0], (from + 1) & 63);
                if (P == 32) {
                    lo |= (uint64_t)(uint32_t)__shfl((int)codes[P / 16 - 1], from & 63) << 32;
                    hi |= (uint64_t)(uint32_t)__shfl((int)codes[P / 16 - 1], (from + 1) & 63) << 32;
                }
                const uint64_t text = o == 0 ? lo : lo >> (2 * o) | hi << (2 * (P - o));
                bool repeats = (P == 32 ? text : text & 0xFFFFFFFFull) == mine;
                if (any_foreign) {
                    const uint64_t f = (uint64_t)(uint32_t)__shfl((int)flags, (from + 1) & 63) << P | (uint32_t)__shfl((int)flags, from & 63);
                    repeats = repeats && (uint32_t)(f >> o & ((1ull << P) - 1ull)) == flags;
                }
                const uint64_t run = __ballot(repeats && lane >= first && lane < row_end && cnt == P) >> first;
                k = __builtin_ctzll(~run);                 // (first > 0, so that bits of zeros were shifted in)
            }
        }
        done = walker;
        if (k == 0) continue;
        if (lane >= first && lane < first + k) {
            int t = (lane - first) * P;
#pragma unroll 1
            for (int i = 10; i >= 0; --i)                  // t % d (t < 64 P <= 2,048)
                if (t >= d << i) t -= d << i;
#pragma unroll 1
            for (int i = 0; i < P; i += 4) {
                Entry v[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int pos = first * P - d + t;     // (behind region `first`: nobody writes there now)
                    v[q] = state[(pos & (P - 1)) * 64 + pos / P];
                    t = t + 1 == d ? 0 : t + 1;
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) state[(i + q) * 64 + lane] = v[q];
            }
        }
        wave_phase();
        done = walker + k;
        if (lane >= walker && lane < done) going = false;
        if (lane == done) {
            going = first + k < row_end && cnt_ahead > 0;
            e = state[(P - 1) * 64 + first + k - 1];
        }
    }
}

// WIDE, P: see above.  PADDED: rows go to their cells of a.pad_ids.  CHUNKS: the items are those of the work
// list (chunks of long rows, then the rows that are one item), a wave each.  CHARS: with the
// single-character ids.
template <bool WIDE, int P, bool CHUNKS, bool CHARS, bool PADDED>
__global__ __launch_bounds__(64 * kAutoMaxWaves) void bpe_auto_kernel(
    BpeArgs a, AutoArgs t, const uint8_t *__restrict__ bytes, const int64_t *__restrict__ offsets,
    BpePlan p, int32_t n_rows, int32_t *__restrict__ tok_tmp, int32_t *__restrict__ lengths)
{
    typedef typename AutoLds<WIDE, P>::Entry Entry;
    static_assert(P == 16 || P == 32, "a region's token starts are the bits of one word");
    static_assert(!CHUNKS || P == 32, "a chunk of 2,048 bytes is a wave");
    // (all of it in one array, the table at its start: an entry and a code are then the next entry's address with one
    // instruction between two reads of the chain)
    extern __shared__ __align__(16) uint8_t smem[];
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int n_waves = (int)blockDim.x >> 6;
    const uint32_t n_entries = 4 * (t.other + 1);
    uint32_t table_bytes = 0;
    const uint32_t tab16 = (n_entries * 2 + 15) / 16, len16 = (t.other + 1 + 15) / 16;
    if (!WIDE) table_bytes = 16 * (tab16 + len16);
    int32_t *const s_longest = reinterpret_cast<int32_t *>(smem + table_bytes + (size_t)n_waves * (64 * P + t.window) * sizeof(Entry));    // [n_waves]
    int32_t *const s_lut = s_longest;                                                                                                     // [256]
    static_assert(!(PADDED && CHARS), "the two share their place");
    const uint8_t *const len_of = smem + (size_t)tab16 * 16;
    const uint32_t *const far_table = reinterpret_cast<const uint32_t *>(t.next);
    Entry *const state = reinterpret_cast<Entry *>(smem + table_bytes) + (size_t)wv * (64 * P + t.window);   // [P][64]
    Entry *const staged = state + 64 * P;                                                                    // [t.window]
    const uint32_t other = WIDE ? (t.other * 4) << 8 | 1u : t.other * 4;

    // (an entry on its way is 32 bits wide, also where one in LDS is 16: as 16 bits every step would clear the others)
    auto step = [&](uint32_t e, uint32_t code) -> uint32_t { return WIDE ? far_table[(e >> 8) + code] : lds_u16(2 * (e + code)); };
    // the same, or `other` if bit `at` of `flags` is set
    auto step_or = [&](uint32_t e, uint32_t code, uint32_t flags, int at) -> uint32_t {
        const uint32_t is = (uint32_t)((int32_t)(flags << (31 - at)) >> 31);
        return (step(e, code) & ~is) | (other & is);
    };
    auto length_of = [&](uint32_t e) -> int { return WIDE ? (int)(e & 0xFFu) : (int)len_of[e >> 2]; };
    auto number_of = [&](uint32_t e) -> uint32_t { return WIDE ? e >> 10 : e >> 2; };

    constexpr int kRowMax = 64 * P;                        // the longest row that a wave takes
    // (list_here) chunk slots and single rows up to and including row 64 q + lane
    constexpr int kListWords = CHUNKS ? kAutoListRows / 64 : 1;
    int32_t slots_to[kListWords], singles_to[kListWords];
    int32_t n_items = t.n_groups, n_mc = 0, n_single0 = 0, n_single1 = 0, n_single2 = 0;
    if (CHUNKS && t.list_here) {
        int64_t from[kListWords], to[kListWords];
#pragma unroll
        for (int q = 0; q < kListWords; ++q) {
            const int row = 64 * q + lane;
            from[q] = to[q] = 0;
            if (row < n_rows) { from[q] = offsets[row]; to[q] = offsets[row + 1]; }
        }
        int32_t n_singles = 0;
#pragma unroll
        for (int q = 0; q < kListWords; ++q) {
            const int64_t len = to[q] - from[q];
            const bool here = 64 * q + lane < n_rows, cut = here && len > p.ext;
            const uint32_t inc = wave_inclusive_sum_u32(cut ? (uint32_t)((len + p.core - 1) / p.core) : 0u);
            const uint64_t single = __ballot(here && !cut);
            slots_to[q] = n_mc + (int32_t)inc;
            singles_to[q] = n_singles + (int32_t)__builtin_amdgcn_mbcnt_hi((uint32_t)(single >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)single, 0u)) +
                            (int32_t)(single >> lane & 1u);
            n_mc = __builtin_amdgcn_readlane(slots_to[q], 63);
            n_singles += (int32_t)__builtin_popcountll(single);
        }
        n_items = n_mc + n_singles;
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            p.counts[0] = n_items;
            p.counts[1] = n_mc;
            p.counts[2] = 0;
            p.counts[3] = 0;
        }
    } else if (CHUNKS) {
        n_mc = p.counts[1];
        n_single0 = p.counts[4];
        n_single1 = p.counts[5];
        n_single2 = p.counts[6];
        n_items = n_mc + n_single0 + (n_single1 + 1) / 2 + (n_single2 + 3) / 4;
    }
    if (WIDE) {
        // A call that follows other kernels finds the table in no L2, and its walks are chains of misses.  The waves that
        // have no item read a word of a line of 128 bytes per lane, the states of the start first (the first twentieth
        // of the 164,729 are every second step), so that the L2 of their XCD has it before the walks have come that far
        // (behind a copy of 512 MB, vocabulary of 32,000: 1,024 rows of 1 KB 23.0 -> 19.4 us, 64 rows 24.9 -> 22.3, 32 of
        // 100 kbp 45.6 -> 43.0; with the table in the L2 1 - 2 % slower).  More workgroups to read all of it: 64 rows
        // of 1 KB 18.3 us, but 13.8 instead of 12.6 with the table in the L2.
        const int32_t busy = n_items <= (int32_t)blockIdx.x ? 0 : (int32_t)((n_items - blockIdx.x + gridDim.x - 1) / gridDim.x);
        if (wv >= busy) {
            const uint32_t line = (blockIdx.x / kXcds * (n_waves - busy) + wv - busy) * 64 + lane;
            uint32_t sum = 0;
            if (32 * line < n_entries) sum = far_table[32 * line];
            asm volatile("" : : "v"(sum));
        }
    }
    if (CHUNKS && t.zero && blockIdx.x == 0 && threadIdx.x == 0) *t.zero = 0;
    int32_t longest = 0;
    // What a wave knows of its item: a chunk (of row `row`, the k-th of nc), or whole rows, one per lane [first, last),
    // with the lanes each of them needs (a region of P bytes to a lane) summed up; they are then taken in as few steps
    // as their lanes fit the wave.
    int32_t item = 0, row_id = 0, k = 0, nc = 1;
    int64_t row_at = 0, row_len = 0;
    int first = 0, last = 0, lanes_to = 0, lanes_own = 0;
    bool chunk = false;
    auto sum_lanes = [&]() {
        lanes_own = 0;
        if (lane >= first && lane < last) lanes_own = row_len <= 0 || row_len > kRowMax ? 1 : ((int)row_len + P - 1) / P;
        lanes_to = (int)wave_inclusive_sum_u32((uint32_t)lanes_own);
    };
    auto take_item = [&](int64_t item64) {
        item = (int32_t)item64;
        k = 0;
        nc = 1;
        int32_t row = 0;
        const int32_t *list = nullptr;
        int32_t list_at = 0;
        const int64_t item_row0 = (int64_t)item * t.rows;
        int item_rows = CHUNKS ? 1 : (int)(n_rows - item_row0 < t.rows ? n_rows - item_row0 : t.rows);
        if (CHUNKS && t.list_here) {
            // the first row whose slots (or single rows) reach beyond the item
            const bool cut = item < n_mc;
            const int32_t want = cut ? item : item - n_mc;
            int32_t before = 0, upto = 0;
            row = -1;
#pragma unroll
            for (int q = 0; q < kListWords; ++q) {
                const int32_t mine = cut ? slots_to[q] : singles_to[q];
                const uint64_t beyond = __ballot(mine > want);
                if (row < 0 && beyond) {
                    const int at = __builtin_ctzll(beyond);
                    row = 64 * q + at;
                    upto = __builtin_amdgcn_readlane(mine, at);
                    if (at > 0) before = __builtin_amdgcn_readlane(mine, at - 1);
                }
                if (row < 0) before = __builtin_amdgcn_readlane(mine, 63);
            }
            if (cut) {
                k = item - before;
                nc = upto - before;
            }
        } else if (CHUNKS && item < n_mc && t.entries_here) {
            // the last row whose first chunk is at or before the item (a row without chunks has its successor's number)
            int32_t lo = 0, hi = n_rows;
            while (hi - lo > 1) {
                const int32_t apart = (hi - lo + 63) >> 6, at = lo + lane * apart;
                const int n = (int)__builtin_popcountll(__ballot(at < hi && p.mc_off[at < hi ? at : lo] <= item));
                lo += (n - 1) * apart;                     // (lane 0 is always at or before it)
                if (lo + apart < hi) hi = lo + apart;
            }
            row = lo;
            const int32_t first_chunk = __builtin_amdgcn_readfirstlane(p.mc_off[row]);
            nc = __builtin_amdgcn_readfirstlane(p.mc_off[row + 1]) - first_chunk;
            k = item - first_chunk;
        } else if (CHUNKS && item < n_mc) {
            const int4 rc = p.rec[item];
            row = __builtin_amdgcn_readfirstlane(rc.x);
            k = __builtin_amdgcn_readfirstlane(rc.y);
            nc = __builtin_amdgcn_readfirstlane(rc.z);
        } else if (CHUNKS) {
            // one single row of the longest class, two of the next, four of the shortest
            int32_t q = item - n_mc, many = 0, of = n_single0;
            list = p.single[0];
            if (q >= n_single0) {
                q -= n_single0; list = p.single[1]; many = 1; of = n_single1;
                if (q >= (n_single1 + 1) / 2) { q -= (n_single1 + 1) / 2; list = p.single[2]; many = 2; of = n_single2; }
            }
            list_at = q << many;
            item_rows = of - list_at < 1 << many ? of - list_at : 1 << many;
        }
        chunk = CHUNKS && nc > 1;
        first = 0;
        last = item_rows;
        row_id = row;
        row_at = 0;
        row_len = 0;
        if (chunk || lane < item_rows) {
            if (!CHUNKS) row_id = (int32_t)(item_row0 + lane);
            else if (list) row_id = list[list_at + lane];
            row_at = offsets[row_id];
            row_len = offsets[row_id + 1] - row_at;
        }
        if (!chunk) sum_lanes();
    };

    // A step: rows [first, first + m) of the item, or the chunk, and what a lane has of it: the row r, that row's lanes
    // lane0 to lane0 + G, and the bytes of its region, [from, from + n) of the batch being what the row (or chunk) has.
    struct Step {
        int m, lane0, G, n;
        bool have;
        int32_t row;
        int64_t start, len, e0, e1;
    };
    auto place = [&]() -> Step {
        Step st;
        st.m = 1;
        st.lane0 = 0;
        st.G = 64;
        st.have = true;
        if (chunk) {
            st.row = row_id;
            st.start = row_at;
            st.len = row_len;
            st.e0 = (int64_t)k * p.core - p.overlap < 0 ? 0 : (int64_t)k * p.core - p.overlap;
            st.e1 = (int64_t)(k + 1) * p.core + p.overlap;
            if (st.e1 > st.len) st.e1 = st.len;
        } else {
            const int lanes_before = first > 0 ? __builtin_amdgcn_readlane(lanes_to, first - 1) : 0;
            const uint64_t in_step = __ballot(lane >= first && lane < last && lanes_to - lanes_before <= 64);
            st.m = (int)__builtin_popcountll(in_step);
            int r = first;
            for (int i = first; i + 1 < first + st.m; ++i)
                if (lane >= __builtin_amdgcn_readlane(lanes_to, i) - lanes_before) r = i + 1;
            st.G = __shfl(lanes_own, r);
            st.lane0 = __shfl(lanes_to, r) - lanes_before - st.G;
            st.have = lane < st.lane0 + st.G;                  // (lanes behind the last row's have none)
            st.start = ((int64_t)__shfl((int)(row_at >> 32), r) << 32) | (uint32_t)__shfl((int)(uint32_t)row_at, r);
            st.len = ((int64_t)__shfl((int)(row_len >> 32), r) << 32) | (uint32_t)__shfl((int)(uint32_t)row_len, r);
            st.row = __shfl(row_id, r);
            st.e0 = 0;
            st.e1 = st.len;
        }
        const bool too_long = st.e1 - st.e0 > kRowMax;         // (longer than the caller declared)
        st.n = st.have && !too_long && st.e1 > st.e0 ? (int)(st.e1 - st.e0) : 0;
        return st;
    };
    auto fetch = [&](const Step &st, auto_u32x4_a1 (&w)[P / 16]) {
        const int s = (lane - st.lane0) * P, cnt = st.n - s;
        const int64_t from = st.start + st.e0 + s;
#pragma unroll
        for (int q = 0; q < P / 16; ++q) {
            w[q] = auto_u32x4_a1{t.letters, t.letters, t.letters, t.letters};
            if (cnt > 16 * q) {
                const uint8_t *const at = bytes + from + 16 * q;
                if (from + 16 * q + 16 <= t.total) {           // (bytes behind the row's end are read, but not behind the batch's)
                    w[q] = *reinterpret_cast<const auto_u32x4_a1 *>(at);
                } else {
                    uint8_t b[16];
#pragma unroll
                    for (int i = 0; i < 16; ++i) b[i] = 16 * q + i < cnt ? at[i] : (uint8_t)0;
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        w[q][i] = (uint32_t)b[4 * i] | ((uint32_t)b[4 * i + 1] << 8) | ((uint32_t)b[4 * i + 2] << 16) | ((uint32_t)b[4 * i + 3] << 24);
                }
            }
        }
    };

    // Whether the first bytes are requested while the tables are staged, and those of an item's next step while a step is
    // worked on.  (Two more copies of the code that does it: forms that stage nothing, or whose waves rarely take more
    // than one step, are 2 - 5 % slower with them.)
    constexpr bool kAhead = !WIDE && P == 32;
    // (neighbouring items go to different CUs, so that a small batch spreads over the chip)
    int64_t item64 = (int64_t)wv * gridDim.x + blockIdx.x;
    Step next{};
    auto_u32x4_a1 ahead_bytes[P / 16];
    // the tables (the transitions and the token lengths), 16 bytes per thread and step
    constexpr int kTablePieces = 6;
    uint4 piece[kAhead ? kTablePieces : 1];
    auto table_piece = [&](uint32_t i) {
        return i < tab16 ? reinterpret_cast<const uint4 *>(t.next)[i] : reinterpret_cast<const uint4 *>(t.len)[i - tab16];
    };
    uint4 *const table_to = reinterpret_cast<uint4 *>(smem);
    if (kAhead) {
#pragma unroll
        for (int q = 0; q < kTablePieces; ++q) {
            const uint32_t i = threadIdx.x + q * blockDim.x;
            if (i < tab16 + len16) piece[q] = table_piece(i);
        }
        if (item64 < n_items) {
            take_item(item64);
            if (first < last) {
                next = place();
                fetch(next, ahead_bytes);
            }
        }
#pragma unroll
        for (int q = 0; q < kTablePieces; ++q) {
            const uint32_t i = threadIdx.x + q * blockDim.x;
            if (i < tab16 + len16) table_to[i] = piece[q];
        }
        for (uint32_t i = threadIdx.x + kTablePieces * blockDim.x; i < tab16 + len16; i += blockDim.x) table_to[i] = table_piece(i);
    } else {
        if (!WIDE) {
            const uint4 *const src = reinterpret_cast<const uint4 *>(t.next), *const src_len = reinterpret_cast<const uint4 *>(t.len);
            for (uint32_t i = threadIdx.x; i < tab16; i += blockDim.x) table_to[i] = src[i];
            for (uint32_t i = threadIdx.x; i < len16; i += blockDim.x) table_to[tab16 + i] = src_len[i];
        }
        item64 -= (int64_t)gridDim.x * n_waves;            // (the loop below begins with the item)
    }
    if (CHARS)
        for (int i = threadIdx.x; i < 256; i += blockDim.x) s_lut[i] = a.char_lut[i];
    if (!WIDE || CHARS) __syncthreads();
    while (item64 < n_items) {
        while (first < last) {                             // (chunks: one step)
            const Step now = next;
            const int m = now.m, lane0 = now.lane0, G = now.G, n = now.n;
            const bool have = now.have;
            const int32_t row = now.row;
            const int64_t start = now.start, len = now.len, e0 = now.e0;
            const int j = lane - lane0;                        // the lane's region within the row
            const int s = j * P;                               // its first byte
            if (chunk && (t.list_here || t.entries_here) && lane == 0) {
                p.rec[item] = make_int4(row, k, nc, (int)len);
                if (t.list_here && k == 0) {
                    p.row_fail[row] = 0;
                    p.mc_off[row] = item;
                }
            }
            const uint8_t *const src = bytes + start + e0;

            // the region's bytes as codes; cnt: how many of its P positions the row has
            const int cnt = n - s < 0 ? 0 : (n - s < P ? n - s : P);
            uint32_t codes[P / 16], flags = 0;
#pragma unroll
            for (int q = 0; q < P / 16; ++q) {
                uint32_t differs;
                codes[q] = letter_codes16(ahead_bytes[q], t.letters, differs);
                if (__ballot(differs != 0)) flags |= foreign16(ahead_bytes[q], t.letters) << (16 * q);      // (few rows hold any)
            }
            // the item's next step begins where this one ends
            const int from = first;
            first += m;
            if (kAhead && !chunk && first < last) {
                next = place();
                fetch(next, ahead_bytes);
            }
            flags &= cnt >= 32 ? ~0u : (1u << cnt) - 1u;                 // (of the positions the row has)
            const bool any_foreign = __ballot(flags != 0) != 0;

            // forward over the own region
            uint32_t e = 0;
            if (any_foreign) {
#pragma unroll
                for (int i = 0; i < P; ++i) {
                    e = step_or(e, (codes[i / 16] >> (2 * (i % 16))) & 3u, flags, i);
                    state[i * 64 + lane] = (Entry)e;
                }
            } else {
#pragma unroll
                for (int i = 0; i < P; ++i) {
                    e = step(e, (codes[i / 16] >> (2 * (i % 16))) & 3u);
                    state[i * 64 + lane] = (Entry)e;
                }
            }
            // and on into the regions to the right until the states are the same, four bytes at a time: once
            // equal they stay equal, so the last of the four tells, and writing equal ones again does no
            // harm (nor does a state behind the row's end, which nothing reads)
            bool going = cnt == P;
            for (int ahead = 1;; ++ahead) {
                const int from = (lane + ahead) & 63;
                uint32_t word = 0, next_word = 0, f2 = 0;
                word = (uint32_t)__shfl((int)codes[0], from);
                if (P == 32) next_word = (uint32_t)__shfl((int)codes[P / 16 - 1], from);
                if (any_foreign) f2 = (uint32_t)__shfl((int)flags, from);
                const int cnt2 = __shfl(cnt, from);
                going = going && j + ahead < G && cnt2 > 0;
                if (!__ballot(going)) break;
                wave_phase();
                if (__builtin_expect(ahead >= kRepeatsFrom / P, 0))
                    copy_repeats<P>(state, codes, flags, any_foreign, cnt, cnt2, lane, lane0, lane0 + G, ahead, e, going);
                for (int i = 0; i < P; i += 4) {
                    if (going) {
                        Entry *const at = state + i * 64 + lane + ahead;
                        const uint32_t there = at[3 * 64];
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            e = step_or(e, (word >> (2 * q)) & 3u, f2, q);
                            at[q * 64] = (Entry)e;
                        }
                        going = e != there;
                    }
                    if (!__ballot(going)) break;
                    word >>= 8;
                    f2 >>= 4;
                    if (P == 32 && i == 12) word = next_word;
                }
            }
            wave_phase();

            // backward: token starts of the region as bits, first from the region's own end
            uint32_t ends = 0;                                 // bit x: a token ends behind the region's byte x
            int entry = s + cnt, entry_end = s + cnt;          // where the walk comes into the region from the right (see border) ...
            int border = s + cnt;                              // ... and where it leaves it: at s, or where the token begins that reaches over s;
            int border_end = s + cnt;                          // that token's end (s itself, if none reaches over)
            const auto token_length = [&](int x) -> int { return length_of(state[x * 64 + lane]); };      // of the token that ends behind byte x
            if (cnt == 0) {                                    // (an empty region: the row ends to its left)
                border = border_end = n;
            } else {
                int x = cnt - 1;
                do {
                    ends |= 1u << x;
                    x -= token_length(x);
                } while (x >= 0);
                border = s + x + 1;
                border_end = x == -1 ? s : s + __builtin_ctz(ends) + 1;
            }
            const bool has_right = cnt > 0 && j + 1 < G && lane < 63;
            int right_end;                                     // end of the token that reaches over the region's end
            for (;;) {
                const int told = __shfl(border, (lane + 1) & 63), told_end = __shfl(border_end, (lane + 1) & 63);
                right_end = has_right ? told_end : s + cnt;
                const bool moved = has_right && (told != entry || told_end != entry_end);
                if (!__ballot(moved)) break;
                if (moved) {
                    entry = told;
                    entry_end = told_end;
                    uint32_t fresh = 0;
                    int x = told - 1 - s;
                    if (x < -1) {                              // one token from left of the region to right of it
                        border = told;
                        border_end = told_end;
                    } else {
                        while (x >= 0 && !(ends >> x & 1u)) {
                            fresh |= 1u << x;
                            x -= token_length(x);
                        }
                        if (x >= 0) {                          // from here on it is the walk made before
                            fresh |= ends & ((2u << x) - 1u);
                        } else {
                            border = s + x + 1;
                            border_end = x == -1 ? s : s + __builtin_ctz(fresh) + 1;
                        }
                    }
                    ends = fresh;
                }
            }
            // token starts of the region: where one ends within it, and at s where none reaches over
            const uint32_t starts = (ends << 1 | (border == s ? 1u : 0u)) & (cnt >= 32 ? ~0u : (1u << cnt) - 1u);

            // every token's number among the wave's
            const uint32_t mine = (uint32_t)__builtin_popcount(starts);
            const uint32_t inc = wave_inclusive_sum_u32(mine);
            const uint32_t before_row = (uint32_t)__shfl((int)inc, lane0 > 0 ? lane0 - 1 : 0);
            const uint32_t base = lane0 > 0 ? before_row : 0u;
            const uint32_t row_last = (uint32_t)__shfl((int)inc, lane0 + G - 1 < 64 ? lane0 + G - 1 : 63);
            const uint32_t n_tok = row_last - base;

            // the region's tokens, last one first: f(number of the token's state -- behind the states: the byte,
            // where it is no letter --, position of its first byte in the region).  Four at a time: their
            // states are read together.
            auto each_token = [&](auto f) {
                uint32_t left = starts;
                int x = right_end - s - 1;                     // the token's last byte, counted from the region's first
                while (left) {
                    int b[4], last[4];
                    bool is[4];
                    uint32_t v[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        is[q] = left != 0;
                        b[q] = 31 - __builtin_clz(left | 1u);
                        last[q] = x;
                        left &= ~(1u << b[q]);
                        x = b[q] - 1;
                    }
                    // (where there is no token any more the place is that of byte -1 or of a byte of the region)
#pragma unroll
                    for (int q = 0; q < 4; ++q) v[q] = number_of(state[(last[q] & (P - 1)) * 64 + lane + (last[q] >> (P == 32 ? 5 : 4))]);
                    if (any_foreign) {
#pragma unroll
                        for (int q = 0; q < 4; ++q)
                            if (is[q] && v[q] == t.other) v[q] = t.other + 1 + src[s + last[q]];
                    }
                    if (WIDE && chunk) {
#pragma unroll
                        for (int q = 0; q < 4; ++q)
                            if (is[q]) v[q] = t.sym[v[q]];
                    }
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        if (is[q]) f(v[q], b[q]);
                }
            };

            if (chunk) {
                // The state's number (wide: the symbol) at every start, kNone elsewhere, and how many start
                // where no neighbour reaches.  A token's number goes to the place of its first byte, whose state
                // no token needs (it is inside one, unless the token is that byte alone).
                each_token([&](uint32_t v, int b) { state[b * 64 + lane] = (Entry)v; });
                int64_t mid_lo = k > 0 ? (int64_t)k * p.core + p.overlap : 0;
                if (mid_lo > len) mid_lo = len;
                const int64_t mid_hi = k + 1 < nc ? (int64_t)(k + 1) * p.core - p.overlap : len;
                uint32_t in_mid = starts;
                const int lo = (int)(mid_lo - e0) - s, hi = (int)(mid_hi - e0) - s;
                if (lo > 0) in_mid &= lo >= 32 ? 0u : ~0u << lo;
                if (hi < 32) in_mid &= hi <= 0 ? 0u : ~0u >> (32 - hi);
                const uint32_t live = wave_inclusive_sum_u32((uint32_t)__builtin_popcount(in_mid));
                if (lane == 63) p.cnt[4 * (size_t)item] = (int32_t)live;
                uint16_t *const raw = p.chunk_sym + (size_t)item * p.ext + s;
#pragma unroll
                for (int i = 0; i < P; i += 8) {
                    uint32_t y[8];
#pragma unroll
                    for (int q = 0; q < 8; ++q) {
                        y[q] = kNone;
                        if (starts >> (i + q) & 1u) {
                            const uint32_t v = state[(i + q) * 64 + lane];
                            y[q] = v;
                        }
                    }
                    if (i < cnt)                               // (a slot is whole vectors: what lies behind the chunk's end is kNone)
                        *reinterpret_cast<uint4 *>(raw + i) = uint4{y[0] | y[1] << 16, y[2] | y[3] << 16, y[4] | y[5] << 16, y[6] | y[7] << 16};
                }
            } else {
                // the step's rows, one per lane again
                int row_tok = 0, row_base = 0;
                {
                    const int at = lanes_to - lanes_own - (from > 0 ? __builtin_amdgcn_readlane(lanes_to, from - 1) : 0);
                    const int at0 = lane >= from && lane < from + m ? at : 0;
                    row_tok = __shfl((int)n_tok, at0);
                    row_base = __shfl((int)base, at0);
                    if (lane >= from && lane < from + m) {
                        lengths[row_id] = row_len > kRowMax ? -1 : row_tok;
                        longest = row_tok > longest ? row_tok : longest;
                    }
                }
                // through LDS, where the wave's tokens fit its window (a token per four bytes always does)
                const bool fits = (uint32_t)__builtin_amdgcn_readlane((int)inc, 63) <= (uint32_t)t.window;
                if (fits) {
                    uint32_t at = inc;
                    each_token([&](uint32_t v, int) { staged[--at] = (Entry)v; });
                    wave_phase();
                }
                if (PADDED) {
                    const int elem = a.pad_elem;
                    if (fits && (a.pad_stride & 3) == 0 && ((uintptr_t)a.pad_ids & (elem >= 4 ? 15 : 4 * elem - 1)) == 0 &&
                        ((uintptr_t)a.pad_mask & 3) == 0) {
                        if (elem == 4) auto_put_rows<4>(a, t.id, staged, row_base, row_tok, from, m, row_id, lane);
                        else if (elem == 8) auto_put_rows<8>(a, t.id, staged, row_base, row_tok, from, m, row_id, lane);
                        else if (elem == 2) auto_put_rows<2>(a, t.id, staged, row_base, row_tok, from, m, row_id, lane);
                        else auto_put_rows<1>(a, t.id, staged, row_base, row_tok, from, m, row_id, lane);
                    } else {
                        // cell by cell: the lanes their own tokens, the row's lanes its padding and mask
                        const int64_t stride = a.pad_stride, at0 = (int64_t)row * stride;
                        const int kept = (int64_t)n_tok < stride ? (int)n_tok : (int)stride;
                        const int64_t shift = a.pad_left ? stride - kept : 0;
                        int at = (int)(inc - base);
                        each_token([&](uint32_t v, int) {
                            --at;
                            if (at < kept) {
                                const int32_t x = t.id[v];
                                auto_put(a.pad_ids, elem, at0 + shift + at, a.pad_remap ? a.pad_remap[x] : x);
                            }
                        });
                        if (have) {
                            for (int64_t c = j; c < stride; c += G) {
                                const bool token = c >= shift && c < shift + kept;
                                if (!token) auto_put(a.pad_ids, elem, at0 + c, a.pad_id);
                                if (a.pad_mask) a.pad_mask[at0 + c] = token ? 1 : 0;
                            }
                        }
                    }
                } else {
                    int32_t *const out = tok_tmp + start;
                    if (fits) {                                // the row's own lanes write its run
                        for (uint32_t c = j; have && c < n_tok; c += G) out[c] = t.id[staged[base + c]];
                    } else {
                        uint32_t at = inc - base;
                        each_token([&](uint32_t v, int) { out[--at] = t.id[v]; });
                    }
                }
            }
            if (CHARS) {
                // the single-character ids of the item's bytes (a chunk: those of its core), by the row's lanes
                int64_t lo = 0, hi = have ? len : 0;
                if (chunk) {
                    lo = (int64_t)k * p.core;
                    hi = (int64_t)(k + 1) * p.core < len ? (int64_t)(k + 1) * p.core : len;
                }
                const int64_t g0 = start + lo, g1 = start + hi;
                const bool quads = ((uintptr_t)a.char_ids & 15) == 0 && ((uintptr_t)a.char_mask & 3) == 0;
                for (int64_t g = (g0 & ~(int64_t)3) + 4 * j; g < g1; g += 4 * G) {
                    if (quads && g >= g0 && g + 4 <= g1) {
                        const uint32_t w = *reinterpret_cast<const auto_u32_a1 *>(bytes + g);
                        const auto_i32x4 v = {s_lut[w & 255u], s_lut[w >> 8 & 255u], s_lut[w >> 16 & 255u], s_lut[w >> 24]};
                        __builtin_nontemporal_store(v, reinterpret_cast<auto_i32x4 *>(a.char_ids + g));
                        if (a.char_mask) __builtin_nontemporal_store(0x01010101u, reinterpret_cast<uint32_t *>(a.char_mask + g));
                    } else {
                        for (int q = 0; q < 4; ++q)
                            if (g + q >= g0 && g + q < g1) {
                                a.char_ids[g + q] = s_lut[bytes[g + q]];
                                if (a.char_mask) a.char_mask[g + q] = 1;
                            }
                    }
                }
            }
            wave_phase();                                      // the wave's part of LDS is rewritten by the next step
            if (!kAhead) break;
        }
        if (!kAhead && first < last) {
            // (rows of the item are left)
        } else {
            item64 += (int64_t)gridDim.x * n_waves;
            if (item64 >= n_items) break;
            take_item(item64);
        }
        if (first < last) {
            next = place();
            fetch(next, ahead_bytes);
        }
    }
    if (PADDED && !CHUNKS && a.max_tree) {
        const uint32_t m = wave_max_u32((uint32_t)longest);
        if (lane == 0) s_longest[wv] = (int32_t)m;
        __syncthreads();
        if (threadIdx.x == 0) {
            int32_t all = 0;
            for (int q = 0; q < n_waves; ++q) all = s_longest[q] > all ? s_longest[q] : all;
            publish_max(a.max_tree, (unsigned)all, a.longest);
        }
    }
}

// A row of many chunks: the tokens of its chunks up to and including each, into the fourth word of their counts.
// The join kernel would otherwise add up, for every chunk, the chunks of its row (padded: all of them, else those in
// front of it), as many reads as the row has chunks squared.  Vocabulary of 4,096, padded: one row of 200 Mbp 16.6 ->
// 0.76 ms (the merge engine 6.1 ms), of 4 Mbp 54.4 -> 43.7 us, of 2 Mbp (1,117 chunks) 32.2 -> 30.6, four of 2 Mbp 58.0 ->
// 57.2; not padded: 200 Mbp 4.35 -> 0.67 ms, 4 Mbp (2,233 chunks) 39.1 -> 37.6, four of 2 Mbp 50.2 -> 53.6.  A workgroup
// looks at kScanRows rows and takes those with as many chunks one after the other, a chunk per thread and step.
__host__ __device__ constexpr int scan_from_chunks(bool padded) { return padded ? 1024 : 2048; }
constexpr int kScanRows = 16;

__global__ __launch_bounds__(1024) void bpe_row_scan_kernel(const int64_t *__restrict__ offsets, int64_t n_rows, int from_chunks, BpePlan p)
{
    __shared__ uint32_t sums[2][16];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int64_t row = (int64_t)blockIdx.x * kScanRows + lane;
    int32_t chunks = 0, first = 0;
    if (lane < kScanRows && row < n_rows) {
        const int64_t len = offsets[row + 1] - offsets[row];
        chunks = len > p.ext ? (int32_t)((len + p.core - 1) / p.core) : 0;
        if (chunks >= from_chunks) first = p.mc_off[row];
    }
    int bank = 0;
    for (uint64_t todo = __ballot(chunks >= from_chunks); todo; todo &= todo - 1) {
        const int at = __builtin_ctzll(todo);              // (the same row in all waves)
        const int32_t nc = __builtin_amdgcn_readlane(chunks, at), m0 = __builtin_amdgcn_readlane(first, at);
        uint32_t before = 0;
        for (int64_t k0 = 0; k0 < nc; k0 += 1024, bank ^= 1) {
            const int64_t k = k0 + threadIdx.x;
            int32_t *const cnt = p.cnt + 4 * ((size_t)m0 + (size_t)k);
            uint32_t c = 0;
            if (k < nc) {
                const int4 part = *reinterpret_cast<const int4 *>(cnt);
                c = (uint32_t)(part.x + (k > 0 ? part.y : 0) + (k + 1 < nc ? part.z : 0));
            }
            const uint32_t inc = wave_inclusive_sum_u32(c);
            if (lane == 63) sums[bank][wv] = inc;
            __syncthreads();                               // (the other bank is read by nobody any more)
            uint32_t to = before + inc;
#pragma unroll
            for (int w = 0; w < 16; ++w) {
                const uint32_t v = sums[bank][w];
                if (w < wv) to += v;
                before += v;
            }
            if (k < nc) cnt[3] = (int32_t)to;
        }
    }
}

// The rows behind the seam kernel: the chunks' tokens put together, a wave per chunk (the chunk is held as in
// bpe_gather_wave_kernel), and the rows that have no seam redone whole.  The two are independent, so they
// share a launch: the first n_slabs workgroups take the rows to be redone (nearly always none), the others
// the chunks.  PADDED: a row goes straight to its cells of a.pad_ids, its padding shared out among its
// chunks; then this launch stands for three (gather, whole rows, padding: 32 rows of 100 kbp, 6.5 + 4.5 +
// 5.3 us).  count_longest: *a.longest (cleared by the kernel in front) becomes the longest row.  SCANNED: the
// row scan kernel has run.
template <bool PADDED, bool SCANNED>
__global__ __launch_bounds__(1024) void bpe_auto_join_kernel(
    BpeArgs a, const int32_t *__restrict__ id, const uint8_t *__restrict__ bytes, const int64_t *__restrict__ offsets, int64_t n_rows,
    int64_t max_len, BpePlan p, int count_longest, int32_t *__restrict__ tok_tmp, int32_t *__restrict__ lengths)
{
    __shared__ __align__(16) uint16_t compact_s[16][kGatherExt];
    const int lane = threadIdx.x & 63;
    if ((int)blockIdx.x < p.n_slabs) {
        if (PADDED && count_longest && blockIdx.x == 0 && threadIdx.x < 64) {      // the rows that were no chunks
            int32_t most = 0;
            for (int64_t row = lane; row < n_rows; row += 64)
                if (offsets[row + 1] - offsets[row] <= p.ext && lengths[row] > most) most = lengths[row];
            const uint32_t m = wave_max_u32((uint32_t)most);
            if (lane == 0) atomicMax(a.longest, (int32_t)m);
        }
        if (p.counts[3] == 0) return;
        uint8_t *const lds = reinterpret_cast<uint8_t *>(compact_s);
        uint32_t *const red = reinterpret_cast<uint32_t *>(lds);
        uint16_t *const b2s = reinterpret_cast<uint16_t *>(lds + 512);
        uint8_t *const D = lds + 1024;
        for (int i = threadIdx.x; i < 256; i += 1024) b2s[i] = a.byte_to_sym[i];
        __syncthreads();
        uint8_t *const slab = p.slabs + (size_t)blockIdx.x * p.slab_bytes;
        const PairTable pt{a.tab, a.shift, a.mul1, a.mul2};
        for (int64_t row = blockIdx.x; row < n_rows; row += p.n_slabs) {
            const int64_t start = offsets[row];
            const int64_t len = offsets[row + 1] - start;
            if (len <= p.ext || !p.row_fail[row]) continue;
            if (len > max_len) {                           // longer than the caller declared: no room in the slab
                if (threadIdx.x == 0) lengths[row] = -1;
            } else {
                const size_t n = ((size_t)len + 7) & ~(size_t)7;
                PosRec<uint32_t> *const P = reinterpret_cast<PosRec<uint32_t> *>(slab);
                uint32_t *const PG = reinterpret_cast<uint32_t *>(P + n);
                uint32_t *const Q = PG + n;
                uint32_t *const C = Q + n / 2;
                bpe_row<1024, uint32_t, 0>(pt, b2s, a.out_remap, bytes + start, (int)len, P, PG, Q, C, D, red, threadIdx.x,
                                           tok_tmp + start, lengths + row);
            }
            __syncthreads();
            if (PADDED) {
                // the row's own workgroup has just written its run and its length
                const int32_t n_tok = __hip_atomic_load(lengths + row, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                const int64_t stride = a.pad_stride, at0 = row * stride;
                const int64_t kept = n_tok < 0 ? 0 : (n_tok < stride ? n_tok : stride), shift = a.pad_left ? stride - kept : 0;
                for (int64_t c = threadIdx.x; c < stride; c += 1024) {
                    const bool token = c >= shift && c < shift + kept;
                    int32_t v = a.pad_id;
                    if (token) {
                        v = __hip_atomic_load(tok_tmp + start + (c - shift), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        if (a.pad_remap) v = a.pad_remap[v];
                    }
                    auto_put(a.pad_ids, a.pad_elem, at0 + c, v);
                    if (a.pad_mask) a.pad_mask[at0 + c] = token ? 1 : 0;
                }
                if (count_longest && threadIdx.x == 0) atomicMax(a.longest, n_tok);
                __syncthreads();
            }
        }
        return;
    }
    const int wv = threadIdx.x >> 6;
    uint16_t *const compact = compact_s[wv];
    const int32_t n_mc = p.counts[1];
    const int64_t n_waves = ((int64_t)gridDim.x - p.n_slabs) * 16;
    for (int64_t m64 = (int64_t)wv * (gridDim.x - p.n_slabs) + (blockIdx.x - p.n_slabs); m64 < n_mc; m64 += n_waves) {
        const int32_t m = (int32_t)m64;
        // first trip: the chunk's symbols and its record
        const uint4 *const src = reinterpret_cast<const uint4 *>(p.chunk_sym + (size_t)m * p.ext);
        uint4 g[4];
#pragma unroll
        for (int q = 0; q < 4; ++q)
            g[q] = lane * 32 + q * 8 < p.ext ? src[lane * 4 + q] : uint4{~0u, ~0u, ~0u, ~0u};
        const int4 rc = p.rec[m];
        const int32_t row = rc.x, k = rc.y, nc = rc.z;
        const int64_t len = rc.w;
        const int64_t e0 = (int64_t)k * p.core - p.overlap < 0 ? 0 : (int64_t)k * p.core - p.overlap;
        // second trip: the seams, the row's state and place, the chunks' counts
        const int32_t seam_l = k > 0 ? p.seam[m - 1] : 0;
        const int32_t seam_r = k + 1 < nc ? p.seam[m] : 0;
        const int32_t failed = p.row_fail[row];
        const int64_t row_at = offsets[row];
        // tokens of the row's chunks in front of this one, and (PADDED) of the whole row
        uint32_t base, n_tok = 0;
        if (SCANNED && nc >= scan_from_chunks(PADDED)) {
            base = k > 0 ? (uint32_t)p.cnt[4 * ((size_t)m - 1) + 3] : 0u;
            if (PADDED) n_tok = (uint32_t)p.cnt[4 * ((size_t)m - k + nc - 1) + 3];
        } else {
            uint32_t before = 0, behind = 0;
            for (int32_t j = lane; j < (PADDED ? nc : k); j += 64) {
                const int4 part = *reinterpret_cast<const int4 *>(p.cnt + 4 * (size_t)(m - k + j));   // {unshared, after left seam, before right seam, -}
                const uint32_t c = (uint32_t)(part.x + (j > 0 ? part.y : 0) + (j + 1 < nc ? part.z : 0));
                if (j < k) before += c; else behind += c;
            }
            base = (uint32_t)__builtin_amdgcn_readlane((int)wave_inclusive_sum_u32(before), 63);
            if (PADDED) n_tok = base + (uint32_t)__builtin_amdgcn_readlane((int)wave_inclusive_sum_u32(behind), 63);
        }
        if (failed) continue;                              // (the same for the whole wave)
        const int64_t lo = k > 0 ? (int64_t)seam_l : 0, hi = k + 1 < nc ? (int64_t)seam_r : len;
        // which of the lane's positions lie in [lo, hi) and start a token
        const int64_t p0 = e0 + lane * 32;
        uint32_t in_span = ~0u;
        if (lo > p0) in_span = lo - p0 >= 32 ? 0u : (~0u << (uint32_t)(lo - p0));
        if (hi < p0 + 32) in_span &= hi <= p0 ? 0u : (~0u >> (uint32_t)(p0 + 32 - hi));
        const uint32_t w[16] = {g[0].x, g[0].y, g[0].z, g[0].w, g[1].x, g[1].y, g[1].z, g[1].w,
                                g[2].x, g[2].y, g[2].z, g[2].w, g[3].x, g[3].y, g[3].z, g[3].w};
        uint32_t live = 0;
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            live |= ((w[q] & 0xFFFFu) != kNone ? 1u : 0u) << (2 * q);
            live |= ((w[q] >> 16) != kNone ? 1u : 0u) << (2 * q + 1);
        }
        live &= in_span;
        const uint32_t mine = (uint32_t)__builtin_popcount(live);
        const uint32_t inc = wave_inclusive_sum_u32(mine);
        const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)inc, 63);
        uint32_t at = inc - mine;
#pragma unroll
        for (int q = 0; q < 32; ++q) {
            if (live >> q & 1u) compact[at++] = (uint16_t)(q & 1 ? w[q >> 1] >> 16 : w[q >> 1] & 0xFFFFu);
        }
        wave_phase();
        if (!PADDED) {
            int32_t *const out = tok_tmp + row_at + base;
#pragma unroll 4
            for (uint32_t t = lane; t < total; t += 64) out[t] = id ? id[compact[t]] : (int32_t)compact[t];
            if (lane == 0 && k + 1 == nc) lengths[row] = (int32_t)(base + total);
        } else {
            const int64_t stride = a.pad_stride, at0 = (int64_t)row * stride;
            const int64_t kept = (int64_t)n_tok < stride ? (int64_t)n_tok : stride, shift = a.pad_left ? stride - kept : 0;
            const int64_t put = kept - (int64_t)base < (int64_t)total ? kept - (int64_t)base : (int64_t)total;
            for (int64_t t = lane; t < put; t += 64) {
                int32_t v = id ? id[compact[t]] : (int32_t)compact[t];
                if (a.pad_remap) v = a.pad_remap[v];
                auto_put(a.pad_ids, a.pad_elem, at0 + shift + base + t, v);
                if (a.pad_mask) a.pad_mask[at0 + shift + base + t] = 1;
            }
            // the chunk's share of the padding
            const int64_t pads = stride - kept, pad0 = a.pad_left ? 0 : kept;
            for (int64_t c = pads * k / nc + lane; c < pads * (k + 1) / nc; c += 64) {
                auto_put(a.pad_ids, a.pad_elem, at0 + pad0 + c, a.pad_id);
                if (a.pad_mask) a.pad_mask[at0 + pad0 + c] = 0;
            }
            if (lane == 0 && k + 1 == nc) {
                lengths[row] = (int32_t)n_tok;
                if (count_longest) atomicMax(a.longest, (int32_t)n_tok);
            }
        }
        wave_phase();                                      // the wave's part of LDS is rewritten by its next chunk
    }
}

}  // namespace dnatok
