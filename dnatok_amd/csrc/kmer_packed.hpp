// Packed k-mer rows in one pass: reads of a few hundred bases, back to back in the output.
// Included by kmer_encode.hip.
//
// Where a row's tokens go depends on the number of tokens of every row in front of it.  A workgroup takes a
// tile of consecutive rows, counts its tokens and publishes the sum; then it adds up what the tiles in front
// of it have published and writes its own tokens.  The sums travel in the caller's out_offsets, in the cell
// behind the tile's last row (the tile's word): kTileOpen until the tile is counted, -1 - its tokens from then
// on (the last tile of a block of sixteen: kBlockSum - the block's tokens), and at last the offset that belongs
// there, which stands for all tiles up to this one.  A tile reads at most fifteen tiles and one word per block
// before its own: with every tile's word read by every later tile, 782 tiles cost more than they saved (the
// words lie a line apart and are read past the L2: 100,000 reads 37.0 us, with blocks and larger tiles 28.3).
//
// (A scan in one pass whose parts look back at those in front of them is Merrill and Garland's decoupled look-back.)
//
// No workgroup depends on another one being on the chip: who finds a word open for too long counts the rows
// behind it itself (their bytes say the same to everybody) and goes on.  It counts only tiles that have published no
// sum of their own, and only until the word comes after all: one row that takes longer than all others would otherwise
// have everybody behind it count the block that it is in (100,000 reads with a row of 200,000 bases in front of them
// 518 us, now 40.6; that row behind them 171, now 45.8).
//
// A row of at most 64 windows (sixteen lanes, kUnitsPerLane windows to a lane) is read once: its windows' codes
// stay in registers from the count to the output, and its few spelled windows in a list in LDS, so that the
// output waits for no load behind its own stores.  Rows of up to twice that are walked by their sixteen lanes,
// longer ones by a wave, from eight steps on by several, once to count and once to write.
//
// What bounds it: trips to memory in a row (the rows' places, their bytes in two batches, the sums, the tokens) with
// the whole batch in flight at once (three workgroups to a CU at 80 registers; at four the compiler spills: 50,000
// reads 29.8 instead of 22.9 us), and vector issue in the count.  Two passes of a launch each for short and for long
// rows with two launches of a scan between them -> one launch behind the one that opens the tiles:
// 100,000 reads of 100 - 300 bp 62.9 -> 28.3 us, 1,000 of them 22.4 -> 11.5, 300,000 139 -> 58, with 50 rows of
// 2 - 20 kbp among 100,000 87.7 -> 41.6, 300 among 3,000 287 -> 31; 20,000 rows of 1,000 bp 42.9 -> 34.9.  With long
// rows shared among a workgroup's waves, on another card: 50 rows of 2 - 20 kbp among 100,000 reads 45.1 -> 31.2 us (the
// two passes 80.9), those 50 in front and all sorted 557 -> 116 (642), a row of 1 Mbp in front 762 -> 128 (578), of
// 5 Mbp 4,176 -> 621 (2,640), ten of 200 kbp 686 -> 280 (1,297); 50,000 rows of 800 - 1,000 bp 66 -> 59 (62).
#pragma once

namespace dnatok {

constexpr int kPackedThreads = 512;                      // 32 groups of sixteen lanes
constexpr int kPackedGroups = kPackedThreads / 16;
constexpr int kPackedHeld = 6;                           // rows of a group that it holds at once, at most,
constexpr int kPackedBatch = 3;                          // and whose bytes are on their way together
constexpr int kPackedRows = kPackedGroups * kPackedHeld; // rows of a tile, at most
constexpr int kPackedPerCu = 3;                          // workgroups of a CU
constexpr int kPackedList = 512;                         // windows spelled by characters that a tile notes for the output
constexpr int kPackedBlock = 16;                         // tiles whose last one publishes the sum of all of them
constexpr int kPackedPolls = 64;                         // trips without an answer until a tile is counted here
constexpr int kPackedStep = 64 * kUnitsPerLane;          // windows of a wave's step in a long row;
constexpr int kPackedParts = kPackedThreads / 64;        // of which there are as many parts, at most,
constexpr int kPackedPart = 4 * kPackedStep;             // of as many windows, at least
constexpr int64_t kTileOpen = INT64_MIN;
constexpr int64_t kBlockSum = -((int64_t)1 << 62);       // minus a block's tokens: its last tile's word

// a value that all lanes of the wave have, as a scalar (what comes out of LDS is not known to be one)
__device__ __forceinline__ int64_t of_wave(int64_t v)
{
    return (int64_t)(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32) | (uint32_t)__builtin_amdgcn_readfirstlane((int)v));
}

// the cell of out_offsets behind tile j's last row
__device__ __forceinline__ int64_t tile_word(int64_t j, int64_t n_rows, int tile_rows)
{
    const int64_t at = (j + 1) * tile_rows;
    return at < n_rows ? at : n_rows;
}

__device__ __forceinline__ int64_t agent_load(const int64_t *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void agent_store(int64_t *p, int64_t v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__global__ __launch_bounds__(256) void kmer_open_tiles_kernel(int64_t *__restrict__ out_offsets, int64_t n_rows, int tile_rows, int64_t n_tiles)
{
    const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (j == 0) out_offsets[0] = 0;
    if (j < n_tiles) out_offsets[tile_word(j, n_rows, tile_rows)] = kTileOpen;
}

template <int K, bool LUT4_LDS>
__global__ __launch_bounds__(kPackedThreads, kPackedPerCu * kPackedThreads / 256) void kmer_packed_kernel(
    KmerArgs a, int all_plain, const uint8_t *__restrict__ bytes, const int64_t *__restrict__ offsets, int64_t n_rows, int tile_rows,
    int polls, int32_t *__restrict__ ids, int64_t *__restrict__ out_offsets, uint8_t *__restrict__ mask,
    int32_t *__restrict__ lengths, int32_t *__restrict__ status)
{
    constexpr uint32_t POW4 = 1u << (2 * K);
    __shared__ int32_t s_single[256];
    __shared__ int32_t s_spell[256];
    __shared__ int32_t s_lut4[LUT4_LDS ? POW4 : 1];
    __shared__ int64_t s_start[kPackedRows + 1];         // where the tile's rows start (the last: end)
    __shared__ uint32_t s_len[kPackedRows];              // their tokens,
    __shared__ int64_t s_to[kPackedRows];                // of them and all rows before them in the tile
    __shared__ uint8_t s_foreign[kPackedRows];
    __shared__ uint32_t s_part[kPackedRows][kPackedParts];   // tokens of a long row's parts
    __shared__ int64_t s_base, s_open;
    __shared__ int64_t s_word[kPackedBlock];
    __shared__ int s_open_tiles, s_came;
    __shared__ unsigned long long s_sum;
    // spelled windows of the held rows: row | first token's place in it << 8, and the characters
    __shared__ uint32_t s_list_at[kPackedList], s_list_lo[kPackedList], s_list_hi[kPackedList];
    __shared__ int s_listed;
    const int lane = threadIdx.x & 63, gl = lane & 15;
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int group = threadIdx.x >> 4;
    const int64_t tile = blockIdx.x;
    const int64_t row0 = tile * tile_rows;
    const int rows = (int)(n_rows - row0 < tile_rows ? n_rows - row0 : tile_rows);

    if ((int)threadIdx.x <= rows) s_start[threadIdx.x] = offsets[row0 + threadIdx.x];
    const int64_t total = offsets[n_rows];
    for (int i = threadIdx.x; i < 256; i += kPackedThreads) {
        const int d = a.digit[i];
        s_single[i] = a.single[i];
        s_spell[i] = a.single[(int)"ACGTN"[d < 0 || d > 4 ? 4 : d]];
    }
    if (LUT4_LDS)
        for (uint32_t i = threadIdx.x; i < POW4; i += kPackedThreads) s_lut4[i] = a.lut4r[i];
    const int32_t *const lut = LUT4_LDS ? s_lut4 : a.lut4r;
    if (threadIdx.x < kPackedRows) {
        s_len[threadIdx.x] = 0;
        s_foreign[threadIdx.x] = 0;
    }
    if (threadIdx.x == 0) {
        s_sum = 0;
        s_came = 0;
        s_listed = 0;
    }
    __syncthreads();

    // rows of at most 64 windows are held; of twice as many they are walked by their sixteen lanes; others by a wave
    const auto held = [](int len) { return len < 65 * K; };
    const auto middling = [](int len) { return len >= 65 * K && len < 129 * K; };

    // A lane's bytes.  (It reads on behind its row's end, but not behind the batch's: only the rows at its very end have to look.)
    const bool roomy = s_start[rows] + kUnitsPerLane * K <= total;
    auto lane_bytes = [&](int64_t pos, bool wanted, uint32_t (&w)[K]) {
        if (roomy) {
#pragma unroll
            for (int q = 0; q < K; ++q) w[q] = 0;
            if (wanted) {
                const LaneBytes<K> all = *reinterpret_cast<const LaneBytes<K> *>(bytes + pos);
#pragma unroll
                for (int q = 0; q < K; ++q) w[q] = all.v[q];
            }
        } else {
            load_lane<K>(bytes, pos, total, wanted, w);
        }
    };
    // Windows [w0, w1) of the row at `at` by the whole wave: f(bytes, their windows, tokens in front of the lane's)
    auto walk = [&](int64_t at, int w0, int w1, bool &foreign_seen, auto f) -> uint32_t {
        uint32_t running = 0;
        bool any = false;
        for (int s0 = w0; s0 < w1; s0 += kPackedStep) {
            const int first = s0 + lane * kUnitsPerLane;
            uint32_t w[K];
            lane_bytes(at + (int64_t)first * K, first < w1, w);
            int32_t slots[kUnitsPerLane];
            bool foreign;
            const uint32_t mine = lane_windows<K>(w, windows_here(w1, first), a.fold, lut, slots, foreign);
            any = any || foreign;
            const uint32_t inc = wave_inclusive_sum_u32(mine);
            f(w, slots, running + inc - mine);
            running += (uint32_t)__builtin_amdgcn_readlane((int)inc, 63);
        }
        foreign_seen = __ballot(any) != 0;
        return running;
    };
    // The rows that are not held nor middling, of which every wave takes its share, those of several parts part by part:
    // f(row, its start and length, the part and its windows [w0, w1)).  (A wave picks its rows out of all by
    // their number: stepping over the others, a few scalar instructions each, took as long as four rows of its own.)
    auto each_long_part = [&](auto f) {
        int turn = 0;
#pragma unroll 1
        for (int i0 = 0; i0 < rows; i0 += 64) {
            int64_t start = 0;
            int len = 0;
            if (i0 + lane < rows) {
                start = s_start[i0 + lane];
                len = (int)(s_start[i0 + lane + 1] - start);
            }
            const bool in_parts = len / K >= 2 * kPackedPart, whole = len >= 129 * K && !in_parts;
            const uint64_t wholes = __ballot(whole);
            const int number = turn + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(wholes >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)wholes, 0u));
            turn += (int)__builtin_popcountll(wholes);
            const auto start_of = [&](int at) {
                return (int64_t)((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(start >> 32), at) << 32 |
                                 (uint32_t)__builtin_amdgcn_readlane((int)start, at));
            };
            for (uint64_t todo = __ballot(whole && (number & (kPackedThreads / 64 - 1)) == wv); todo; todo &= todo - 1) {
                const int at = __builtin_ctzll(todo), n = __builtin_amdgcn_readlane(len, at);
                f(i0 + at, start_of(at), n, 0, 0, n / K);
            }
            for (uint64_t todo = __ballot(in_parts); todo; todo &= todo - 1) {
                const int at = __builtin_ctzll(todo), n = __builtin_amdgcn_readlane(len, at), full = n / K;
                const int most = full / kPackedPart, parts = most > kPackedParts ? kPackedParts : most;
                const int each = ((full - 1) / parts / kPackedStep + 1) * kPackedStep;
#pragma unroll 1
                for (int part = 0; part < parts; ++part, ++turn) {
                    if ((turn & (kPackedThreads / 64 - 1)) != wv) continue;
                    const int w0 = part * each < full ? part * each : full;
                    f(i0 + at, start_of(at), n, part, w0, full - w0 < each ? full : w0 + each);
                }
            }
        }
    };
    // count (the long rows first, before the others' codes take the registers)
    each_long_part([&](int i, int64_t at, int n, int part, int w0, int w1) {
        bool foreign;
        const uint32_t count = walk(at, w0, w1, foreign, [](const uint32_t (&)[K], const int32_t (&)[kUnitsPerLane], uint32_t) {});
        if (lane == 0) {
            s_part[i][part] = count;
            atomicAdd(&s_len[i], count + (uint32_t)(part == 0 ? n % K : 0));
            if (foreign) s_foreign[i] = 1;
        }
    });
    const int sets = tile_rows / kPackedGroups;          // rows of a group
    uint32_t codes[kPackedHeld][kUnitsPerLane / 2];      // of the lane's windows, two to a word
    uint8_t kinds[kPackedHeld];                          // which of them are spelled (four bits) | how many there are << 4
    uint16_t from[kPackedHeld];                          // tokens of the row in front of the lane's
    uint8_t tail_byte[kPackedHeld];                      // a trailing character (lanes below the tail's length)
#pragma unroll
    for (int r0 = 0; r0 < kPackedHeld; r0 += kPackedBatch) {
        if (r0 >= sets) break;
        // The bytes of a batch of rows first, so that they are one trip to memory.
        uint32_t w[kPackedBatch][K];
#pragma unroll
        for (int b = 0; b < kPackedBatch; ++b) {
            const int r = r0 + b, i = r * kPackedGroups + group;
            const int64_t start = i < rows ? s_start[i] : 0;
            const int len = i < rows ? (int)(s_start[i + 1] - start) : 0;
            const bool here = held(len) && gl * kUnitsPerLane * K + K <= len;
            const int64_t pos = start + gl * (kUnitsPerLane * K);
            lane_bytes(pos, here, w[b]);
            tail_byte[r] = 0;
            if (gl < len % K) tail_byte[r] = bytes[start + len - len % K + gl];
        }
#pragma unroll
        for (int b = 0; b < kPackedBatch; ++b) {
            const int r = r0 + b, i = r * kPackedGroups + group;
            const int len = i < rows ? (int)(s_start[i + 1] - s_start[i]) : 0;
            const int full = held(len) ? len / K : 0;
            const int n_win = windows_here(full, gl * kUnitsPerLane);
            bool foreign;
            uint32_t code[kUnitsPerLane];
            uint32_t spelled = lane_codes<K>(w[b], n_win, a.fold, code, foreign);
            if (!all_plain) {
#pragma unroll
                for (int j = 0; j < kUnitsPerLane; ++j)
                    if (j < n_win && lut[code[j]] < 0) spelled |= 1u << j;
            }
            codes[r][0] = code[0] | code[1] << 16;
            codes[r][1] = code[2] | code[3] << 16;
            kinds[r] = (uint8_t)(spelled | (uint32_t)n_win << 4);
            const uint32_t mine = (uint32_t)n_win + (K - 1) * (uint32_t)__builtin_popcount(spelled);
            const uint32_t inc = row16_inclusive_sum(mine);
            from[r] = (uint16_t)(inc - mine);
            const uint32_t bad = (uint32_t)(__ballot(foreign) >> (lane & 48)) & 0xFFFFu;
            if (i < rows && held(len) && gl == 15) {
                s_len[i] = inc + (uint32_t)(len % K);
                s_foreign[i] = bad ? 1 : 0;
            }
            if (spelled) {
                uint32_t at = inc - mine;
#pragma unroll
                for (int j = 0; j < kUnitsPerLane; ++j) {
                    if (spelled >> j & 1u) {
                        const int e = atomicAdd(&s_listed, 1);
                        if (e < kPackedList) {
                            uint32_t c[2] = {0, 0};
#pragma unroll
                            for (int q = 0; q < K; ++q) {
                                const int bi = j * K + q;
                                c[q >> 2] |= ((w[b][bi >> 2] >> (8 * (bi & 3))) & 255u) << (8 * (q & 3));
                            }
                            s_list_at[e] = (uint32_t)i | at << 8;
                            s_list_lo[e] = c[0];
                            s_list_hi[e] = c[1];
                        }
                    }
                    at += spelled >> j & 1u ? K : 1;
                }
            }
        }
    }
    // what put_plain and put_spelled take of a held row
    auto windows_of = [&](int r, int32_t (&win)[kUnitsPerLane]) {
        int32_t id[kUnitsPerLane];
#pragma unroll
        for (int j = 0; j < kUnitsPerLane; ++j) id[j] = lut[codes[r][j >> 1] >> (16 * (j & 1)) & 0xFFFFu];
#pragma unroll
        for (int j = 0; j < kUnitsPerLane; ++j) win[j] = j >= kinds[r] >> 4 ? kNothing : kinds[r] >> j & 1 ? kSpelled : id[j];
    };
    // A group's middling rows, one after the other, in step with the wave's other groups: f(row, its start, the lane's
    // bytes, their windows, tokens in front of the lane's); g(row, start, length, its tokens, whether it has foreign bytes)
    auto each_middling_row = [&](auto f, auto g) {
#pragma unroll 1
        for (int r = 0; r < sets; ++r) {
            const int i = r * kPackedGroups + group;
            const int64_t start = i < rows ? s_start[i] : 0;
            const int len = i < rows ? (int)(s_start[i + 1] - start) : 0;
            const bool is = middling(len);
            if (!__ballot(is)) continue;
            const int full = is ? len / K : 0;
            uint32_t running = 0;
            bool any = false;
#pragma unroll 1
            for (int s0 = 0; s0 < 128; s0 += 64) {
                const int first = s0 + gl * kUnitsPerLane;
                uint32_t w[K];
                lane_bytes(start + (int64_t)first * K, first < full, w);
                int32_t slots[kUnitsPerLane];
                bool foreign;
                const uint32_t mine = lane_windows<K>(w, windows_here(full, first), a.fold, lut, slots, foreign);
                any = any || foreign;
                const uint32_t inc = row16_inclusive_sum(mine);
                if (is) f(i, w, slots, running + inc - mine);
                running += row16_last(inc);
            }
            const uint32_t bad = (uint32_t)(__ballot(any) >> (lane & 48)) & 0xFFFFu;
            if (is) g(i, start, len, running + (uint32_t)(len % K), bad != 0);
        }
    };
    each_middling_row([](int, const uint32_t (&)[K], const int32_t (&)[kUnitsPerLane], uint32_t) {},
                      [&](int i, int64_t, int, uint32_t count, bool foreign) {
                          if (gl == 0) {
                              s_len[i] = count;
                              s_foreign[i] = foreign ? 1 : 0;
                          }
                      });
    __syncthreads();

    // A row's tokens and those of all rows before it in the tile; the tile's sum is published, and the sums in front of
    // it are added up, by the first wave: those of the tiles before it in its block, and of the blocks before that one,
    // back to the first word that stands for everything in front of it.
    const int in_block = (int)(tile % kPackedBlock);
    const int64_t block = tile / kPackedBlock;
    const bool last = in_block == kPackedBlock - 1;
    int64_t own = 0, siblings = 0, sum = 0;              // (first wave) tokens of the tile, of those before it in its block, of what lies before the block
    int64_t end = block;                                 // (first wave) blocks [0, end) are still to be added
    bool have_siblings = false;
    if (wv == 0) {
        constexpr int kPer = kPackedRows / 64;
        uint32_t v[kPer];
        uint64_t mine = 0;
#pragma unroll
        for (int q = 0; q < kPer; ++q) {
            v[q] = kPer * lane + q < rows ? s_len[kPer * lane + q] : 0u;
            mine += v[q];
        }
        uint64_t inc = mine;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint64_t x = __shfl_up(inc, d);
            if (lane >= d) inc += x;
        }
        uint64_t to = inc - mine;
#pragma unroll
        for (int q = 0; q < kPer; ++q) {
            to += v[q];
            s_to[kPer * lane + q] = (int64_t)to;
        }
        own = (int64_t)__shfl(inc, 63);
        if (lane == 0 && !last) agent_store(out_offsets + tile_word(tile, n_rows, tile_rows), -1 - own);
    }
    const auto sum_of_lanes = [](int64_t v) {
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d);
        return v;
    };
    for (;;) {
        // (rows [open0, open1), whose sum nobody has published, and what it is to be published as)
        if (wv == 0) {
            int64_t open = -1;                           // the first tile of the rows, or -1: all is known
            int open_tiles = 0;
            for (int tries = 0; !have_siblings || end > 0;) {
                // lanes below kPackedBlock - 1: the tiles before this one; the others: the last blocks
                constexpr int kBlocksFrom = kPackedBlock - 1;
                int64_t word = 0;
                const int64_t b = end - 1 - (lane - kBlocksFrom);
                const int64_t j = lane < kBlocksFrom ? block * kPackedBlock + lane : (b + 1) * kPackedBlock - 1;
                if (lane < kBlocksFrom ? lane < in_block && !have_siblings : b >= 0)
                    word = agent_load(out_offsets + tile_word(j, n_rows, tile_rows));
                const uint64_t is_open = __ballot(word == kTileOpen);
                const int64_t had = end;
                const bool had_siblings = have_siblings;
                if (!have_siblings && !(is_open & ((1ull << kBlocksFrom) - 1ull))) {
                    // (a tile that has already put its final word there: all up to it is in that word)
                    const uint64_t done = __ballot(lane < in_block && word >= 0);
                    const int from = done ? 63 - __builtin_clzll(done) : -1;
                    siblings = sum_of_lanes(lane >= in_block || lane < from ? 0 : lane == from ? word : -1 - word);
                    have_siblings = true;
                    if (done) {
                        sum = 0;
                        end = 0;
                    }
                    if (last && lane == 0 && !done) agent_store(out_offsets + tile_word(tile, n_rows, tile_rows), kBlockSum - siblings - own);
                }
                if (had == end && end > 0) {
                    const uint64_t all_open = is_open >> kBlocksFrom;
                    const uint64_t is_all = __ballot(word >= 0) >> kBlocksFrom;      // (in front of the first block: 0 stands for all)
                    const int stop = all_open ? __builtin_ctzll(all_open) : 64 - kBlocksFrom;
                    const int upto = is_all ? __builtin_ctzll(is_all) : 64 - kBlocksFrom;
                    const int at = lane - kBlocksFrom;
                    if (at >= 0 && at < stop && at < upto) sum += kBlockSum - word;
                    if (upto < stop) {
                        if (at == upto) sum += word;
                        end = 0;
                    } else {
                        end -= stop;
                    }
                }
                if ((!have_siblings || end > 0) && had == end && had_siblings == have_siblings && ++tries > polls) {
                    open_tiles = 1;
                    if (!have_siblings) open = block * kPackedBlock + __builtin_ctzll(is_open);
                    else { open = (end - 1) * kPackedBlock; open_tiles = kPackedBlock; }
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
            }
            const int64_t before = sum_of_lanes(sum) + siblings;
            if (lane == 0) {
                s_open = open;
                s_open_tiles = open_tiles;
                s_base = before;
                if (open < 0) agent_store(out_offsets + tile_word(tile, n_rows, tile_rows), before + own);
            }
            if (lane < open_tiles) s_word[lane] = agent_load(out_offsets + (open + lane + 1) * tile_rows);      // (never the batch's last tile)
        }
        __syncthreads();
        const int64_t open = of_wave(s_open);
        if (open < 0) break;
        // Nobody has published the sum of these tiles: the tokens of the rows of those whose own is not known either, a row
        // to a wave, for as long as the word that is waited for does not come.
        const int open_tiles = __builtin_amdgcn_readfirstlane(s_open_tiles);
        int64_t *const awaited = out_offsets + (open + open_tiles) * tile_rows;
        bool came = false;
        for (int q = 0; q < open_tiles && !came; ++q) {
            const int64_t word = of_wave(s_word[q]);
            if (word < 0 && word > kBlockSum) {
                if (threadIdx.x == 0) atomicAdd(&s_sum, (unsigned long long)(-1 - word));
                continue;
            }
            for (int i = wv; i < tile_rows && !came; i += kPackedThreads / 64) {
                const int64_t row = (open + q) * tile_rows + i, at = of_wave(offsets[row]);
                const int n = (int)(of_wave(offsets[row + 1]) - at), full = n / K;
                // (a byte at a time: the held rows' codes have the registers)
                uint32_t count = lane == 0 ? (uint32_t)(n % K) : 0u;
#pragma unroll 1
                for (int w0 = 0; w0 < full && !came; w0 += 64) {
                    came = __builtin_amdgcn_readfirstlane(agent_load(awaited) == kTileOpen ? 0 : 1) != 0;
                    if (w0 + lane >= full) continue;
                    uint32_t code = 0, odd = 0;
#pragma unroll 1
                    for (int b = 0; b < K; ++b) {
                        const uint32_t v = bytes[at + (int64_t)(w0 + lane) * K + b], d = v >> 1 & 3u;
                        odd |= (v ^ (0x47544341u >> (8 * d) & 255u)) & a.fold & 255u;
                        code |= d << (2 * b);
                    }
                    count += odd || lut[code] < 0 ? K : 1;
                }
                count = wave_inclusive_sum_u32(count);
                if (lane == 63) atomicAdd(&s_sum, (unsigned long long)count);
            }
        }
        if (came && lane == 0) s_came = 1;
        __syncthreads();
        if (threadIdx.x == 0) {
            if (!s_came) {
                const int64_t word = open_tiles == 1 ? -1 - (int64_t)s_sum : kBlockSum - (int64_t)s_sum;
                atomicCAS(reinterpret_cast<unsigned long long *>(awaited), (unsigned long long)kTileOpen, (unsigned long long)word);
            }
            s_sum = 0;
            s_came = 0;
        }
    }

    // out
    const int64_t base = s_base;
    const auto put_plain = [&](int32_t *out, const int32_t (&win)[kUnitsPerLane]) {      // out: the lane's first token
        if ((win[0] | win[1] | win[2] | win[3]) >= 0) {
            *reinterpret_cast<int4v_a4 *>(out) = int4v_a4{win[0], win[1], win[2], win[3]};
        } else {
            int at = 0;
#pragma unroll
            for (int j = 0; j < kUnitsPerLane; ++j) {
                if (win[j] >= 0) out[at] = win[j];
                at += win[j] == kSpelled ? K : 1;
            }
        }
    };
    const auto put_spelled = [&](int32_t *out, const uint32_t (&b)[K], const int32_t (&win)[kUnitsPerLane]) {
        int at = 0;
#pragma unroll
        for (int j = 0; j < kUnitsPerLane; ++j) {
            if (win[j] == kSpelled) {
#pragma unroll
                for (int q = 0; q < K; ++q) {
                    const int bi = j * K + q;
                    out[at + q] = s_spell[(b[bi >> 2] >> (8 * (bi & 3))) & 255u];
                }
            }
            at += win[j] == kSpelled ? K : 1;
        }
    };
    const int listed = s_listed;
#pragma unroll
    for (int r = 0; r < kPackedHeld; ++r) {
        const int i = r * kPackedGroups + group;
        if (i >= rows) continue;
        const int len = (int)(s_start[i + 1] - s_start[i]), tail = len % K;
        if (!held(len)) continue;
        int32_t *const end = ids + base + s_to[i], *const out = end - s_len[i] + from[r];
        int32_t win[kUnitsPerLane];
        windows_of(r, win);
        put_plain(out, win);
        if (gl < tail) end[gl - tail] = s_single[tail_byte[r]];
    }
    if (listed <= kPackedList) {
        for (int e = threadIdx.x; e < listed; e += kPackedThreads) {
            const uint32_t at = s_list_at[e], c[2] = {s_list_lo[e], s_list_hi[e]};
            const int i = at & 255u;
            int32_t *const out = ids + base + s_to[i] - s_len[i] + (at >> 8);
#pragma unroll
            for (int q = 0; q < K; ++q) out[q] = s_spell[(c[q >> 2] >> (8 * (q & 3))) & 255u];
        }
    } else {
        // (more than the list has room for: the bytes once more)
#pragma unroll
        for (int r = 0; r < kPackedHeld; ++r) {
            const int i = r * kPackedGroups + group;
            if (i >= rows || !held((int)(s_start[i + 1] - s_start[i]))) continue;
            uint32_t b[K];
            int32_t win[kUnitsPerLane];
            windows_of(r, win);
            lane_bytes(s_start[i] + gl * (kUnitsPerLane * K), win[0] != kNothing, b);
            put_spelled(ids + base + s_to[i] - s_len[i] + from[r], b, win);
        }
    }
    each_middling_row(
        [&](int i, const uint32_t (&b)[K], const int32_t (&win)[kUnitsPerLane], uint32_t at) {
            int32_t *const out = ids + base + s_to[i] - s_len[i] + at;
            put_plain(out, win);
            put_spelled(out, b, win);
        },
        [&](int i, int64_t start, int len, uint32_t, bool) {
            const int tail = len % K;
            if (gl < tail) (ids + base + s_to[i])[gl - tail] = s_single[bytes[start + len - tail + gl]];
        });
    each_long_part([&](int i, int64_t start, int len, int part, int w0, int w1) {
        int32_t *const end = ids + base + of_wave(s_to[i]);
        uint32_t before = 0;
        for (int q = 0; q < part; ++q) before += s_part[i][q];
        before = (uint32_t)__builtin_amdgcn_readfirstlane((int)before);
        int32_t *const first = end - s_len[i] + before;
        // (the trailing characters are requested in front of the walk: behind its stores they are another trip)
        const int tail = part == 0 ? len % K : 0;
        const uint8_t tail_at = lane < tail ? bytes[start + len - tail + lane] : (uint8_t)0;
        bool foreign;
        walk(start, w0, w1, foreign, [&](const uint32_t (&b)[K], const int32_t (&win)[kUnitsPerLane], uint32_t at) {
            put_plain(first + at, win);
            put_spelled(first + at, b, win);
        });
        if (lane < tail) end[lane - tail] = s_single[tail_at];
    });
    if ((int)threadIdx.x < rows) {
        const int i = threadIdx.x;
        lengths[row0 + i] = (int32_t)s_len[i];
        if (status) status[row0 + i] = s_foreign[i] ? DNATOK_ROW_INVALID_BYTE : 0;
        // (the last one's cell has been written; its neighbours in memory belong to the words of other tiles)
        if (i + 1 < rows) agent_store(out_offsets + row0 + i + 1, base + s_to[i]);
    }
    if (mask) {
        const int64_t n_tok = s_to[rows - 1];
        uint8_t *const m = mask + base;
        const int64_t head = (16 - (int64_t)(reinterpret_cast<uintptr_t>(m) & 15)) & 15, lo = head < n_tok ? head : n_tok;
        const int64_t hi = lo + ((n_tok - lo) & ~(int64_t)15);
        if ((int64_t)threadIdx.x < lo) m[threadIdx.x] = 1;
        for (int64_t c = lo + 16 * (int64_t)threadIdx.x; c < hi; c += 16 * kPackedThreads)
            *reinterpret_cast<uint4 *>(m + c) = uint4{0x01010101u, 0x01010101u, 0x01010101u, 0x01010101u};
        if (hi + (int64_t)threadIdx.x < n_tok) m[hi + threadIdx.x] = 1;
    }
}

}  // namespace dnatok
