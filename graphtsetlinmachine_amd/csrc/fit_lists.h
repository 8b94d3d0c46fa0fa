// What the training kernels share: a clause as a list of rows, Type I feedback bits a byte per lane, and the
// feedback of one automaton word from masks of classes.
//
// A training step evaluates every clause on one graph, but feedback moves few automata across the middle, so a
// clause's include plane is nearly always what it was a step ago.  The rows that a clause ANDs are therefore kept as
// a list in LDS - 16-bit row numbers, the node-type row first, then the included literals - and the list is made anew
// only when the clause's include plane has changed.  A row of a graph of a few hundred nodes is a dozen words: a lane
// reads two words at a time, the wave's lanes are groups of 2^lg lanes, as many as a row takes, and every group
// reads rows of its own, eight per batch; the groups' results are ANDed at the end.  Bound by the latency of
// two dependent LDS reads per batch: 50 literals on 12 words are one batch of eight groups, where walking the include
// plane's set bits on the scalar unit, eight rows at a time with 12 of 64 lanes at work, took seven round trips.
#pragma once

constexpr int FITL_BATCH_LOG = 3;  // rows that a group reads per batch, as a power of two: one 128-bit read of row numbers

// log2 of the lanes that a row of `words` words takes (at most 64 words, two to a lane, at least 8 lanes)
inline int fitl_lanes_log(int words) { return words <= 16 ? 3 : words <= 32 ? 4 : 5; }
// words between two rows in LDS: whole pairs
__host__ __device__ inline int fitl_stride(int words) { return (words + 1) & ~1; }
// entries of a list that holds every literal: whole batches
inline int fitl_entries(int literals, int lg) {
    const int batch = 1 << (FITL_BATCH_LOG + 6 - lg);
    return (literals + 1 + batch - 1) / batch * batch;
}

// v ANDed over the wave's groups of 2^lg lanes (lg 3, 4 or 5); every lane gets its place's result.
__device__ __forceinline__ uint32_t fitl_and_groups(uint32_t v, int lg) {
    if (lg <= 3) v &= (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x128, 0xF, 0xF, true);  // row_ror 8
    if (lg <= 4) {
        const auto s = __builtin_amdgcn_permlane16_swap(v, v, false, false);  // even and odd rows of 16 lanes, each doubled
        v = s[0] & s[1];
    }
    const auto s = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return s[0] & s[1];
}

// the number of bits of m below this lane's
__device__ __forceinline__ int fitl_lanes_below(unsigned long long m) {
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// v summed over this lane and those below it (no memory access, six instructions)
__device__ __forceinline__ int fitl_sum_up_to(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);  // row_shr 1, 2, 4, 8: within rows of 16 lanes
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);  // row_bcast 15 into rows 1 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);  // row_bcast 31 into rows 2 and 3
    return v;
}

// One wave adds 64 include words to a clause's list, lane w holding word `first` / 32 + w in `mine` (0 where there is none):
// row `first` + 32 w + b for every set bit b.  The list holds n entries; entries from `cap` on are counted, not
// written.  Returns the new n.  A word pair is the mask of the lanes that write: no memory is read.
__device__ __forceinline__ int fitl_append(uint32_t mine, int words, int first, uint16_t *list, int cap, int n, int lane) {
    for (int w = 0; w < words; w += 2) {
        unsigned long long m = (uint32_t)__builtin_amdgcn_readlane(mine, w);
        if (w + 1 < words) m |= (unsigned long long)(uint32_t)__builtin_amdgcn_readlane(mine, w + 1) << 32;
        const int j = n + fitl_lanes_below(m);
        if (((m >> lane) & 1ull) && j < cap) list[j] = (uint16_t)(first + 32 * w + lane);
        n += __popcll(m);
    }
    return n;
}
// ... and fills up the last batch with the all-ones row.
__device__ __forceinline__ void fitl_finish(uint16_t *list, int cap, int n, int ones_row, int lg, int lane) {
    const int batch = 1 << (FITL_BATCH_LOG + 6 - lg), full = min(cap, (n + batch - 1) & ~(batch - 1));
    for (int j = n + lane; j < full; j += 64) list[j] = (uint16_t)ones_row;
}

// The AND of the `n` rows of a list (n >= 1; the list 16-byte aligned): words 2 L and 2 L + 1 in lane L of every group of
// lanes.  col: the lane's first word of row 0, 8-byte aligned; rows are `stride` words apart.
__device__ __forceinline__ uint2 fitl_truth(const uint16_t *list, int n, const uint32_t *col, int stride, int lg, int lane) {
    const int groups_log = 6 - lg;
    const uint4 *at = reinterpret_cast<const uint4 *>(list) + (lane >> lg);
    int batches = (n - 1) >> (FITL_BATCH_LOG + groups_log);  // after the first
    uint2 acc = make_uint2(0xFFFFFFFFu, 0xFFFFFFFFu);
    auto row = [&](uint32_t r) { return *reinterpret_cast<const uint2 *>(col + r * (uint32_t)stride); };
    uint4 rows = at[0];
    for (;;) {
        uint4 ahead = rows;
        at += 1 << groups_log;
        if (batches > 0) ahead = at[0];
        const uint2 r[8] = {row(rows.x & 0xFFFFu), row(rows.x >> 16), row(rows.y & 0xFFFFu), row(rows.y >> 16),
                            row(rows.z & 0xFFFFu), row(rows.z >> 16), row(rows.w & 0xFFFFu), row(rows.w >> 16)};
#pragma unroll
        for (int u = 0; u < 8; ++u) acc.x &= r[u].x, acc.y &= r[u].y;
        if (batches == 0) break;
        // (false everywhere stays false; not worth asking ahead of the last batch)
        if (batches > 1 && __ballot((fitl_and_groups(acc.x, lg) | fitl_and_groups(acc.y, lg)) != 0u) == 0ull) break;
        --batches;
        rows = ahead;
    }
    return make_uint2(fitl_and_groups(acc.x, lg), fitl_and_groups(acc.y, lg));
}

// The same for a clause whose literals exceed its list: the include plane's set bits (word w at inc[w * inc_stride]), every group of
// lanes on words of its own, eight rows at a time: 400 nodes, 4,000 clauses of 960 literals 16.8 us per example, 38.9 with all groups
// on the same word.
__device__ __forceinline__ uint2 fitl_walk(const uint32_t *inc, int inc_stride, int LA, uint32_t filter, int type_row, int ones_row,
                                           const uint32_t *col, int stride, int lg, int lane) {
    auto row = [&](int r) { return *reinterpret_cast<const uint2 *>(col + r * stride); };
    uint2 acc = row(type_row);
    for (int w0 = 0; w0 < LA; w0 += 64 >> lg) {
        const int w = w0 + (lane >> lg);
        uint32_t m = w < LA ? inc[w * inc_stride] : 0u;
        if (w == LA - 1) m &= filter;
        if (__ballot(m != 0u) == 0ull) continue;
        if (__ballot((fitl_and_groups(acc.x, lg) | fitl_and_groups(acc.y, lg)) != 0u) == 0ull) return make_uint2(0u, 0u);
        while (__ballot(m != 0u) != 0ull) {
            uint2 r[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                r[u] = row(m ? 32 * w + __builtin_ctz(m) : ones_row);
                m &= m - 1;
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) acc.x &= r[u].x, acc.y &= r[u].y;
        }
    }
    return make_uint2(fitl_and_groups(acc.x, lg), fitl_and_groups(acc.y, lg));
}

// The truth of a clause at a graph's nodes from the AND of its rows: lane L of the first group keeps nodes 64 L .. 64 L + 63, the
// others keep none.
__device__ __forceinline__ uint2 fitl_nodes(uint2 acc, const FitGraph &fg, int lg, int lane) {
    const bool mine = lane < (1 << lg);
    return make_uint2(mine && 2 * lane < fg.words ? (acc.x >> fg.shift) & fg.mask : 0u, mine && 2 * lane + 1 < fg.words ? acc.y : 0u);
}

// The node a clause learns from (K7): the (random * count >> 32)-th of the nodes it is true at, lane L holding nodes
// 64 L .. 64 L + 63; -1: none.  One wave; the same result in every lane.
__device__ __forceinline__ int fitl_pick_node(uint2 v, uint32_t random, int lane) {
    const int own = __popc(v.x) + __popc(v.y), up_to = fitl_sum_up_to(own);
    const uint32_t count = (uint32_t)__builtin_amdgcn_readlane(up_to, 63);
    if (count == 0u) return -1;
    const int pick = (int)(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane(random) * count) >> 32);
    const int from = __ffsll((long long)__ballot(pick < up_to)) - 1;
    const unsigned long long word = (unsigned long long)(uint32_t)__builtin_amdgcn_readlane(v.y, from) << 32 | (uint32_t)__builtin_amdgcn_readlane(v.x, from);
    const int nth = pick - (__builtin_amdgcn_readlane(up_to, from) - __popcll(word));
    return 64 * from + __ffsll((long long)(__ballot(fitl_lanes_below(word) == nth) & word)) - 1;
}

// A quarter of gtm_feedback_bits: bits 8 q .. 8 q + 7, one generator call.  A word's four calls, one after the other in one
// lane, are a chain of 600 instructions while most lanes have nothing to draw.
__device__ __forceinline__ uint32_t fitl_feedback_byte(uint32_t k0, uint32_t k1, uint32_t clause, uint32_t word, uint32_t q, uint32_t step,
                                                       uint32_t bank, uint32_t class_id, uint32_t threshold16) {
    if (threshold16 >= 65536u) return 0xFFu;
    const philox_out r = philox4x32_10(clause, word * 4u + q, step, GTM_TAG_FEEDBACK | (bank << 8) | (class_id << 16), k0, k1);
    uint32_t bits = 0u;
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
        bits |= (uint32_t)((r.v[i] & 0xFFFFu) < threshold16) << (i * 2u);
        bits |= (uint32_t)((r.v[i] >> 16) < threshold16) << (i * 2u + 1u);
    }
    return bits;
}

// Type I feedback of the classes in `pos`, Type II of those in `neg` (32 classes from class `first` on), in the order of the classes, on
// one automaton word (kernels.py:141-183, and :98-139 for message banks).  fb_of[k]: Type I bits of class k.
template <int MAXB, bool EXACT>
__device__ __forceinline__ void fitl_feedback(fits_word<MAXB, EXACT> &word, uint32_t pos, uint32_t neg, bool fired, bool learns, int boost,
                                              uint32_t x, const uint32_t *fb_of) {
    for (uint32_t m = pos | neg; m; m &= m - 1) {
        const int k = __builtin_ctz(m);
        uint32_t up = fired ? ~x & ~word.top() : 0u, down = 0u;
        if ((pos >> k) & 1u) {
            const uint32_t fb = fb_of[k];
            up = learns ? (boost == 1 ? x : x & ~fb) : 0u;
            down = learns ? ~x & fb : fb;
        }
        word.count(up, down);
    }
}
