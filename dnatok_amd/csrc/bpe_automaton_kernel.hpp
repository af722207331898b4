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
// (L2: 164,729 states are 2.6 MB), the waves' share of LDS alone.
//
// Every phase is a chain of dependent reads, so what a launch takes is the number of waves in flight.
// Sixteen share the table instead of eight since a wave's tokens leave through a window of one per four
// bytes (more than that are written lane by lane) and a chunk's go where the states were: 16,384 rows of
// 1 KB 54.7 -> 29.2 us, 100,000 reads 123 -> 57 us.  (That includes the walk into the next region four bytes
// at a time, comparing the last of the four, and the padded rows of a wave written as one run of cells.)
//
// Per call, the merge engine -> the automaton: 1,024 rows of 1 KB 29.4 -> 11.7 us, 16,384 of them 236.5 ->
// 29.2 us, 100,000 reads of 100 - 300 bp (int64 rows) 349 -> 57 us, 4,096 ragged reads of 12 Mbp 253.5 ->
// 83.9 us (all with the vocabulary of 4,096), 32 rows of 100 kbp (32,000) 143.8 -> 74.3 us.
#pragma once

namespace dnatok {

struct AutoArgs {
    const void *next;            // narrow: uint16 [4 * (n_states + 1)], entry = 4 * state; wide: uint32, entry = 4 * state << 8 | length
    const uint8_t *len;          // [n_states + 1] (narrow)
    const uint16_t *sym;         // [n_states + 1 + 256] token of a state; behind the states: symbol of a byte
    const int32_t *id;           // the same through the table's out_remap
    uint32_t other;              // the state behind a byte that is no letter; its successors are the row start's
    uint32_t letters;            // the letters by code (bits 1 and 2 of the byte)
    int32_t lanes, rows;         // lanes per row, rows per wave (lanes * rows <= 64)
    int32_t n_groups;            // whole rows: n_rows / rows, rounded up (chunks: the work list says)
    int32_t window;              // tokens a wave has room for on their way out
    int64_t total;               // bytes of the batch
};

// Waves of a workgroup, which has a CU to itself: as many as the LDS holds, at most sixteen (four per SIMD).
constexpr int kAutoMaxWaves = 16;
constexpr uint32_t kAutoNarrowStates = 10400;    // the most the narrow form has LDS for, beside the waves' share
constexpr size_t kAutoLdsBytes = 163840 - 1152;  // what a workgroup may take: the CU's, less the static arrays (1,088 bytes)

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
        const size_t w = (kAutoLdsBytes - table_bytes(n_states)) / (state_bytes + least_window * sizeof(Entry));
        return w > (size_t)kAutoMaxWaves ? kAutoMaxWaves : (int)w;
    }
    static int window(uint32_t n_states)
    {
        const size_t w = ((kAutoLdsBytes - table_bytes(n_states)) / waves(n_states) - state_bytes) / sizeof(Entry) & ~(size_t)7;
        return w > (size_t)(64 * P) ? 64 * P : (int)w;
    }
    static size_t bytes(uint32_t n_states)
    {
        return table_bytes(n_states) + waves(n_states) * (state_bytes + window(n_states) * sizeof(Entry));
    }
};

// Between two phases of a wave's work on its LDS: what a lane wrote before is what the others read after.
__device__ __forceinline__ void wave_phase()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Codes of the 16 bytes of w (two bits each, the first byte lowest) and the bytes that are no letters.
__device__ __forceinline__ uint32_t letter_codes16(const auto_u32x4_a1 w, uint32_t letters, uint32_t &foreign)
{
    uint32_t codes = 0, bad = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const uint32_t sel = (w[q] >> 1) & 0x03030303u;
        const uint32_t back = __builtin_amdgcn_perm(letters, letters, sel);
        const uint32_t two = sel | (sel >> 6);
        codes |= ((two | (two >> 12)) & 0xFFu) << (8 * q);
        // the high bit of every byte that differs, then four bits together
        const uint32_t d = back ^ w[q];
        const uint32_t hi = ((d & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | d;
        const uint32_t f = (hi >> 7) & 0x01010101u;
        bad |= ((f | (f >> 7) | (f >> 14) | (f >> 21)) & 0xFu) << (4 * q);
    }
    foreign = bad;
    return codes;
}

// One id, in the padded output's own integer width.
__device__ __forceinline__ void auto_put(void *ids, int elem, int64_t at, int32_t v)
{
    if (elem == 4) reinterpret_cast<int32_t *>(ids)[at] = v;
    else if (elem == 8) reinterpret_cast<int64_t *>(ids)[at] = (int64_t)v;
    else if (elem == 2) reinterpret_cast<int16_t *>(ids)[at] = (int16_t)v;
    else reinterpret_cast<uint8_t *>(ids)[at] = (uint8_t)v;
}

// The rows [row0, row0 + rows) of the padded output, whose tokens lie in `staged`: row r's n_tok tokens
// from `base` on, both known to lane r * G.  The rows are taken as one run of cells, four to a lane
// (they start on such a boundary).
template <int ELEM, typename Entry>
__device__ __forceinline__ void auto_put_rows(const BpeArgs &a, const int32_t *id, const Entry *staged, int base, int n_tok,
                                              int G, int rows, int64_t row0, int lane)
{
    const int stride = (int)a.pad_stride, quads = stride >> 2;
    const int64_t n_steps = ((int64_t)rows * quads + 63) >> 6;
    int r = 0, c = lane;
    for (int64_t step = 0; step < n_steps; ++step, c += 64) {
        while (c >= quads && r < rows) { c -= quads; ++r; }
        const int from = (r < rows ? r : 0) * G;
        const int n = __shfl(n_tok, from), b = __shfl(base, from);
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
            const int64_t at = (row0 + r) * stride + 4 * c;
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
    extern __shared__ __align__(16) uint8_t smem[];
    __shared__ int32_t s_longest[PADDED ? kAutoMaxWaves : 1];
    __shared__ int32_t s_lut[CHARS ? 256 : 1];
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int n_waves = (int)blockDim.x >> 6;
    const uint32_t n_entries = 4 * (t.other + 1);
    uint32_t table_bytes = 0;
    if (!WIDE) {
        // the transition table and the token lengths, 16 bytes per thread and step
        const uint32_t tab16 = (n_entries * 2 + 15) / 16, len16 = (t.other + 1 + 15) / 16;
        const uint4 *const src = reinterpret_cast<const uint4 *>(t.next);
        uint4 *const dst = reinterpret_cast<uint4 *>(smem);
        for (uint32_t i = threadIdx.x; i < tab16; i += blockDim.x) dst[i] = src[i];
        const uint4 *const src_len = reinterpret_cast<const uint4 *>(t.len);
        for (uint32_t i = threadIdx.x; i < len16; i += blockDim.x) dst[tab16 + i] = src_len[i];
        table_bytes = 16 * (tab16 + len16);
    }
    if (CHARS)
        for (int i = threadIdx.x; i < 256; i += blockDim.x) s_lut[i] = a.char_lut[i];
    const uint16_t *const table = reinterpret_cast<const uint16_t *>(smem);
    const uint8_t *const len_of = smem + (size_t)((n_entries * 2 + 15) / 16) * 16;
    const uint32_t *const far_table = reinterpret_cast<const uint32_t *>(t.next);
    Entry *const state = reinterpret_cast<Entry *>(smem + table_bytes) + (size_t)wv * (64 * P + t.window);   // [P][64]
    Entry *const staged = state + 64 * P;                                                                    // [t.window]
    const Entry other = WIDE ? (Entry)((t.other * 4) << 8 | 1u) : (Entry)(t.other * 4);
    __syncthreads();

    auto step = [&](Entry e, uint32_t code) -> Entry {
        if (WIDE) return (Entry)far_table[((uint32_t)e >> 8) + code];
        return (Entry)table[(uint32_t)e + code];
    };
    auto length_of = [&](Entry e) -> int {
        if (WIDE) return (int)((uint32_t)e & 0xFFu);
        return (int)len_of[(uint32_t)e >> 2];
    };
    auto number_of = [&](Entry e) -> uint32_t { return WIDE ? (uint32_t)e >> 10 : (uint32_t)e >> 2; };

    const int G = t.lanes, R = t.rows;
    const int r = lane / G, j = lane - r * G;              // the lane's row within the wave, and its region within the row
    const int s = j * P;                                   // first byte of the region
    const int lane0 = lane - j;                            // the row's first lane
    const int cap = G * P;
    const int32_t n_items = CHUNKS ? p.counts[0] : t.n_groups;
    const int32_t n_mc = CHUNKS ? p.counts[1] : 0;
    const int32_t n_single0 = CHUNKS ? p.counts[4] : 0, n_single1 = CHUNKS ? p.counts[5] : 0;
    int32_t longest = 0;
    // (neighbouring items go to different CUs, so that a small batch spreads over the chip)
    for (int64_t item64 = (int64_t)wv * gridDim.x + blockIdx.x; item64 < n_items; item64 += (int64_t)gridDim.x * n_waves) {
        const int32_t item = (int32_t)item64;
        int32_t row = 0, k = 0, nc = 1;
        bool have = true;
        if (CHUNKS) {
            if (item < n_mc) {
                const int4 rc = p.rec[item];
                row = rc.x; k = rc.y; nc = rc.z;
            } else {
                int32_t q = item - n_mc;
                const int32_t *list = p.single[0];
                if (q >= n_single0) {
                    q -= n_single0; list = p.single[1];
                    if (q >= n_single1) { q -= n_single1; list = p.single[2]; }
                }
                row = list[q];
            }
            row = __builtin_amdgcn_readfirstlane(row);
            k = __builtin_amdgcn_readfirstlane(k);
            nc = __builtin_amdgcn_readfirstlane(nc);
        } else {
            row = item * R + r;
            have = r < R && row < n_rows;
            if (!have) row = n_rows - 1;
        }
        const int64_t start = offsets[row];
        const int64_t len = offsets[row + 1] - start;
        int64_t e0 = 0, e1 = len;
        if (CHUNKS && nc > 1) {
            e0 = (int64_t)k * p.core - p.overlap < 0 ? 0 : (int64_t)k * p.core - p.overlap;
            e1 = (int64_t)(k + 1) * p.core + p.overlap;
            if (e1 > len) e1 = len;
        }
        const bool too_long = e1 - e0 > cap;
        const int n = have && !too_long && e1 > e0 ? (int)(e1 - e0) : 0;
        const uint8_t *const src = bytes + start + e0;

        // the region's bytes as codes; cnt: how many of its P positions the row has
        const int cnt = n - s < 0 ? 0 : (n - s < P ? n - s : P);
        uint32_t codes[P / 16], flags = 0;
#pragma unroll
        for (int q = 0; q < P / 16; ++q) {
            auto_u32x4_a1 w = {0, 0, 0, 0};
            if (cnt > 16 * q) {
                const uint8_t *const at = src + s + 16 * q;
                if (start + e0 + s + 16 * q + 16 <= t.total) {       // (bytes behind the row's end are read, but not behind the batch's)
                    w = *reinterpret_cast<const auto_u32x4_a1 *>(at);
                } else {
                    uint8_t b[16];
#pragma unroll
                    for (int i = 0; i < 16; ++i) b[i] = 16 * q + i < cnt ? at[i] : (uint8_t)0;
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        w[i] = (uint32_t)b[4 * i] | ((uint32_t)b[4 * i + 1] << 8) | ((uint32_t)b[4 * i + 2] << 16) | ((uint32_t)b[4 * i + 3] << 24);
                }
            }
            uint32_t foreign;
            codes[q] = letter_codes16(w, t.letters, foreign);
            flags |= foreign << (16 * q);
        }
        flags &= cnt >= 32 ? ~0u : (1u << cnt) - 1u;                 // (of the positions the row has)
        const bool any_foreign = __ballot(flags != 0) != 0;

        // forward over the own region
        Entry e = 0;
        if (any_foreign) {
#pragma unroll
            for (int i = 0; i < P; ++i) {
                e = step(e, (codes[i / 16] >> (2 * (i % 16))) & 3u);
                if (flags >> i & 1u) e = other;
                state[i * 64 + lane] = e;
            }
        } else {
#pragma unroll
            for (int i = 0; i < P; ++i) {
                e = step(e, (codes[i / 16] >> (2 * (i % 16))) & 3u);
                state[i * 64 + lane] = e;
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
            for (int i = 0; i < P; i += 4) {
                if (going) {
                    Entry *const at = state + i * 64 + lane + ahead;
                    const Entry there = at[3 * 64];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        e = step(e, (word >> (2 * q)) & 3u);
                        if (any_foreign && (f2 >> q & 1u)) e = other;
                        at[q * 64] = e;
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
        auto state_at = [&](int pos) -> Entry { return state[(pos & (P - 1)) * 64 + lane0 + pos / P]; };
        uint32_t starts = 0;
        int entry = s + cnt, entry_end = s + cnt;          // where the walk comes into the region from the right (see border) ...
        int border = s + cnt;                              // ... and where it leaves it: at s, or where the token begins that reaches over s;
        int border_end = s + cnt;                          // that token's end (s itself, if none reaches over)
        if (cnt == 0) border = border_end = n;
        {
            int pos = s + cnt;
            while (pos > s) {
                border_end = pos;
                pos -= length_of(state[(pos - 1 - s) * 64 + lane]);
                if (pos >= s) starts |= 1u << (pos - s);
            }
            if (cnt > 0) border = pos;                     // (an empty region: the row ends to its left)
            if (cnt > 0 && pos == s) border_end = s;
        }
        const bool has_right = cnt > 0 && j + 1 < G && lane < 63;
        int right_end;                                     // end of the token that reaches over the region's end
        for (;;) {
            const int told = __shfl(border, (lane + 1) & 63), told_end = __shfl(border_end, (lane + 1) & 63);
            right_end = has_right ? told_end : s + cnt;
            const bool moved = has_right && (told != entry || told_end != entry_end);
            if (moved) { entry = told; entry_end = told_end; }
            if (moved && told < s) {                       // one token from left of the region to right of it
                starts = 0;
                border = told;
                border_end = told_end;
            } else if (moved) {
                uint32_t fresh = 0;
                int pos = told, end = told_end;
                for (;;) {
                    if (pos - s < cnt) {
                        const uint32_t bit = 1u << (pos - s);
                        if (starts & bit) {                // from here on it is the walk made before
                            fresh |= starts & (bit | (bit - 1u));
                            break;
                        }
                        fresh |= bit;
                    }
                    if (pos > s) {
                        end = pos;
                        pos -= length_of(state[(pos - 1 - s) * 64 + lane]);
                    } else {
                        end = s;
                    }
                    if (pos <= s) {
                        if (pos == s) {
                            fresh |= 1u;
                            end = s;
                        }
                        border = pos;
                        border_end = end;
                        break;
                    }
                }
                starts = fresh;
            }
            if (!__ballot(moved)) break;
        }

        // every token's number among the wave's
        const uint32_t mine = (uint32_t)__builtin_popcount(starts);
        const uint32_t inc = wave_inclusive_sum_u32(mine);
        const uint32_t before_row = (uint32_t)__shfl((int)inc, lane0 > 0 ? lane0 - 1 : 0);
        const uint32_t base = lane0 > 0 ? before_row : 0u;
        const uint32_t row_last = (uint32_t)__shfl((int)inc, lane0 + G - 1 < 64 ? lane0 + G - 1 : 63);
        const uint32_t n_tok = row_last - base;
        const bool chunk = CHUNKS && nc > 1;

        // the region's tokens, last one first: f(number of the token's state -- behind the states: the byte,
        // where it is no letter --, position of its first byte in the region)
        auto each_token = [&](auto f) {
            uint32_t left = starts;
            int end = right_end;
            while (left) {
                const int b = 31 - __builtin_clz(left);
                left ^= 1u << b;
                uint32_t v = number_of(state_at(end - 1));
                if (any_foreign && v == t.other) v = t.other + 1 + src[end - 1];
                end = s + b;
                f(v, b);
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
                        y[q] = WIDE ? (uint32_t)t.sym[v] : v;
                    }
                }
                if (i < cnt)                               // (a slot is whole vectors: what lies behind the chunk's end is kNone)
                    *reinterpret_cast<uint4 *>(raw + i) = uint4{y[0] | y[1] << 16, y[2] | y[3] << 16, y[4] | y[5] << 16, y[6] | y[7] << 16};
            }
        } else {
            if (j == 0 && have) {
                lengths[row] = too_long ? -1 : (int32_t)n_tok;
                longest = (int32_t)n_tok > longest ? (int32_t)n_tok : longest;
            }
            // through LDS, where the wave's tokens fit its window (a token per four bytes always does)
            const bool fits = (uint32_t)__builtin_amdgcn_readlane((int)inc, 63) <= (uint32_t)t.window;
            if (fits) {
                uint32_t at = inc;
                each_token([&](uint32_t v, int) { staged[--at] = (Entry)v; });
                wave_phase();
            }
            if (PADDED) {
                const int64_t row0 = (int64_t)item * R;
                const int rows = n_rows - row0 < R ? (int)(n_rows - row0) : R;
                const int elem = a.pad_elem;
                if (fits && (a.pad_stride & 3) == 0 && ((uintptr_t)a.pad_ids & (elem >= 4 ? 15 : 4 * elem - 1)) == 0 &&
                    ((uintptr_t)a.pad_mask & 3) == 0) {
                    if (elem == 4) auto_put_rows<4>(a, t.id, staged, (int)base, (int)n_tok, G, rows, row0, lane);
                    else if (elem == 8) auto_put_rows<8>(a, t.id, staged, (int)base, (int)n_tok, G, rows, row0, lane);
                    else if (elem == 2) auto_put_rows<2>(a, t.id, staged, (int)base, (int)n_tok, G, rows, row0, lane);
                    else auto_put_rows<1>(a, t.id, staged, (int)base, (int)n_tok, G, rows, row0, lane);
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
                    for (uint32_t c = j; c < n_tok; c += G) out[c] = t.id[staged[base + c]];
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
        wave_phase();                                      // the wave's part of LDS is rewritten by its next item
    }
    if (PADDED && a.max_tree) {
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

}  // namespace dnatok
