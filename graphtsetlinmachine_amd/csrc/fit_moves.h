// A whole run of training examples (the loop at tm.py:669-747) of a model WITH message layers in one cooperative
// launch, for data sets whose edges are a few moves (score_moves.h: chains, grids): an edge goes from node n to n + d
// and has type t, and few (t, d) occur.
//
// The exchange is that of fit_deep_persistent.h: per message layer every workgroup ORs into the received rows what its
// own clauses make the nodes receive, one device-wide wait, every workgroup copies all received rows into LDS; at
// the end the class sums.  What differs:
//   - what a clause makes the nodes receive along a move is its truth row shifted by d, where an edge of the move
//     ends: no edge is staged or walked;
//   - clauses are lists of rows per bank (fit_lists.h), remade when an include plane changes.  A message literal's
//     row is the received row, negated literals their complements: lists are octets of one sign;
//   - where a clause's words fit its share of the workgroup's 16 waves, its automata live in the lanes' registers for the
//     whole run and every one of its waves decides its feedback for itself (REGS); else they stay in memory and the words
//     of the clauses that get feedback are shared out;
//   - random words of the gates and of the next node pick are drawn, and the words of the picked nodes fetched, while
//     the class sums travel.
// Bound by the two or three device-wide exchanges per example (few clauses), or by the generator calls of the Type I
// feedback and the copies of the received rows (thousands of clauses).  us per example, edges walked and clauses' include
// planes walked (fit_deep_persistent.h) -> here: 1,000-node chains, 200 clauses 20.5 -> 11 to 11.7; chains of 10 to 40 nodes, 333 clauses,
// three layers 26 -> 15.7; 324-node grids, 2,000 clauses, three layers of 1,024 bits 55 -> 27.6 (256 bits: 21.5); 841-node grids, 8,000
// clauses, three layers 170 -> 61, of which the slowest workgroup's evaluation, for which all others waited, was more than half.
#pragma once

constexpr int FITM_MAX_CLASSES = 64;
constexpr int FITM_REGS_CLASSES = 63;  // lane 63 draws for the node pick
constexpr int FITM_CHUNK = 4096;  // examples of a launch, for which the moves' masks are kept

struct FitMovesParams {
    // data set
    const uint32_t *tiles, *X, *node_index, *n_nodes;
    const int32_t *encoded_Y;
    TileGeom tg;
    int first_example, n_examples;
    uint32_t first_step;
    TileMoves moves;
    const uint32_t *masks;  // [example of the launch][moves.n][S] nodes where an edge of the move ends
    // model
    uint32_t *bank[GTM_MAX_DEPTH];
    int32_t *weights;
    const uint32_t *hv;
    int depth, literals, n_types, C, LA, MC, MW, M, MB, B, K, T, negative, boost, max_included;
    uint32_t filter, thr16[GTM_MAX_DEPTH], k0, k1;
    uint64_t q_thr;
    // exchange (device memory, zero on entry)
    uint32_t *got;                  // [3][depth - 1][M][S]
    uint32_t *vec;                  // [depth - 2][max_nodes][MW] what each node received, node-major (all layers but the last)
    unsigned long long *arrived;    // [depth - 1][FITD_PARTS * FITD_STRIDE]
    unsigned long long *class_sum;  // [3][K][FITP_SUM_PARTS] words FITP_SUM_STRIDE apart
    uint32_t *abort_flag;
    uint32_t spin_limit;
    unsigned long long wait_ticks;
    int force_abort;
    int clauses_per_group;
    const int *perm;     // as in fit_deep_persistent.h
    uint16_t *lists;     // [workgroups][clauses_per_group][list0 + (depth - 1) * listm], unless REGS: in LDS
    int S, lanes_log;    // words between rows, log2 of the lanes that a row takes
    int rows_words;      // LDS words of one graph's layer-0 rows (ROWS_LDS)
    int list0, listm;    // entries of the list of bank 0 and of a message bank, whole octets
    int max_nodes;
};

// Do a workgroup's clauses send to so many rows that they meet in them?  ORed into memory one by one, the rows of short messages
// were a queue of all clauses: us per example with the edges walked, ORed in memory, ORed in LDS first (chains of 20 nodes,
// two moves, two bits a message): 20,000 clauses, 32-bit messages (316 rows sent by a workgroup) 90, 108, 31; 5,000 clauses, 32 bits
// 36, 37, 22, 256 bits (80 rows) 34, 22.6, 21.0; 8,000 clauses, 1,024 bits, 100 nodes (128 rows) 79, 48, 50.  Automata in memory only: in
// registers a workgroup has at most 16 clauses, which are ahead of the walk without (4,000 clauses, 32 bits 32 and 29).  A kernel of
// its own: the choice inside one cost calls that do not collect up to 4 %.
inline bool fit_moves_collects(int own, int n_moves, int MB, int M) { return 4 * (int64_t)own * n_moves * MB > M; }

inline size_t fit_moves_lds_words(bool regs, bool rows_lds, int depth, int own, int LA, int MC, int MB, int M, int K, int S, int rows_words,
                                  int list0, int listm, int n_moves) {
    const size_t o = (size_t)own, words = (size_t)LA + (size_t)(depth - 1) * MC;
    return (size_t)M * S + (rows_lds ? 2 * (size_t)rows_words : 0) + (regs ? o * (list0 + (depth - 1) * listm) / 2 : 0) + o * S +
           2 * (size_t)n_moves * S + o * words + 3 * o * K + 4 * o + 4 * o * depth + 6 * o + o * n_moves * MB + o * (MC / 2);
}

// masks[example][move][S]: the nodes where an edge of the move ends.  One workgroup per example; LDS: n * S words.
__global__ void k_fit_move_masks(const uint32_t *__restrict__ n_nodes, const uint32_t *__restrict__ node_index,
                                 const uint32_t *__restrict__ n_edges, const uint32_t *__restrict__ edge_index,
                                 const uint32_t *__restrict__ edge, int first_example, const uint32_t *__restrict__ header, int n_moves, int S,
                                 uint32_t *__restrict__ masks) {
    extern __shared__ uint32_t ends[];  // [n_moves][S]
    for (int i = threadIdx.x; i < n_moves * S; i += blockDim.x) ends[i] = 0u;
    __syncthreads();
    const int ex = first_example + (int)blockIdx.x;
    const uint32_t n = n_nodes[ex];
    const int64_t base = node_index[ex];
    for (uint32_t v = threadIdx.x; v < n; v += blockDim.x) {
        const uint32_t count = n_edges[base + v];
        const uint2 *out_edges = reinterpret_cast<const uint2 *>(edge) + edge_index[base + v];
        for (uint32_t e = 0; e < count; ++e) {
            const uint2 to = out_edges[e];
            const uint32_t key = tile_move_key(v, to.x, to.y, n);
            for (int k = 0; k < n_moves; ++k)
                if (key && key == header[k]) atomicOr(&ends[k * S + (to.x >> 5)], 1u << (to.x & 31u));
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < n_moves * S; i += blockDim.x) masks[(int64_t)blockIdx.x * n_moves * S + i] = ends[i];
}

// Two words that need not lie on an 8-byte boundary (rows in a tile).
struct __attribute__((packed, aligned(4))) fitm_pair {
    uint32_t x, y;
};

// acc ANDed with the rows of the octets part * G + group, (part + parts) * G + group, ... of a list of n8 octets, G groups of
// lanes; an octet whose first entry has bit 15 set holds rows to be complemented (SIGNED).  An octet that is not there is
// the last one again: an AND twice is an AND once.  Afterwards every group's acc is its own.
template <bool SIGNED, typename Pair, typename Col>
__device__ __forceinline__ uint2 fitm_rows(uint2 acc, const uint4 *list, int n8, int part, int parts, Col col, int stride, int lg, int lane) {
    const int groups = 64 >> lg, group = lane >> lg;
    auto row = [&](uint32_t r) {
        const Pair v = *reinterpret_cast<const Pair *>(col + r * (uint32_t)stride);
        return make_uint2(v.x, v.y);
    };
    int at = part * groups;
    if (at >= n8) return acc;
    uint4 rows = list[min(at + group, n8 - 1)];
    for (;;) {
        const int next = at + parts * groups;
        uint4 ahead = rows;
        if (next < n8) ahead = list[min(next + group, n8 - 1)];
        constexpr uint32_t MASK = SIGNED ? 0x7FFFu : 0xFFFFu;
        const uint32_t flip = SIGNED ? 0u - ((rows.x >> 15) & 1u) : 0u;
        const uint2 r[8] = {row(rows.x & MASK), row((rows.x >> 16) & MASK), row(rows.y & MASK), row((rows.y >> 16) & MASK),
                            row(rows.z & MASK), row((rows.z >> 16) & MASK), row(rows.w & MASK), row((rows.w >> 16) & MASK)};
#pragma unroll
        for (int u = 0; u < 8; ++u) acc.x &= r[u].x ^ flip, acc.y &= r[u].y ^ flip;
        if (next >= n8) return acc;
        // (false everywhere stays false; not worth asking ahead of the last octets)
        if (next + parts * groups < n8 && __ballot((fitl_and_groups(acc.x, lg) | fitl_and_groups(acc.y, lg)) != 0u) == 0ull) return make_uint2(0u, 0u);
        at = next;
        rows = ahead;
    }
}

// MAXB, EXACT: the planes of an automaton (fits_word).  REGS: automata in registers, lists in LDS.  ROWS_LDS: the graph's layer-0 rows
// are staged in LDS; else they are read from the tile in place.  COLLECT (not REGS): what the workgroup's clauses send is ORed in LDS first.
template <int MAXB, bool EXACT, bool REGS, bool ROWS_LDS, bool COLLECT>
__global__ __launch_bounds__(FITP_BLOCK) void k_fit_moves(FitMovesParams p) {
    extern __shared__ __align__(16) uint32_t lds[];
    __shared__ int32_t votes[64], sums[64], labels[2][64];
    __shared__ int go_on, n_own_shared, n_busy, n_stale, next_unit, next_words;
    constexpr int WAVES = FITP_BLOCK / 64, POLL = WAVES - 1;  // the last wave announces, adds and polls
    int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int G = (int)gridDim.x, g = (int)blockIdx.x, own_max = p.clauses_per_group;
    const int LA = p.LA, MC = p.MC, MW = p.MW, M = p.M, B = EXACT ? MAXB : p.B, K = p.K, S = p.S, depth = p.depth, L = depth - 1, NM = p.moves.n;
    const int words_all = LA + L * MC;   // automaton words of a clause over all banks
    const int lg = p.lanes_log;
    const int list_entries = p.list0 + L * p.listm;

    // LDS carve-up
    static_assert(!(REGS && COLLECT), "");
    uint32_t *mrows = lds;                                              // [M][S] received rows of the current layer
    uint32_t *rows_both = mrows + (size_t)M * S;                        // ROWS_LDS: [2][rows_words] layer-0 rows of this and the next graph
    uint32_t *lists_lds = rows_both + (ROWS_LDS ? 2 * p.rows_words : 0);  // REGS: [own][list_entries] 16-bit entries
    uint32_t *truth = lists_lds + (REGS ? (size_t)own_max * list_entries / 2 : 0);  // [own][S]
    uint32_t *ends = truth + (size_t)own_max * S;                       // [2][NM][S] where the moves of this and the next graph end
    uint32_t *inc = ends + 2 * NM * S;                                  // [own][words_all] include planes
    int32_t *wts = (int32_t *)(inc + (size_t)own_max * words_all);      // [own][K]
    uint32_t *gate = (uint32_t *)(wts + (size_t)own_max * K);           // [own][K][2] random words of the feedback gates
    uint32_t *type1 = gate + 2 * (size_t)own_max * K;                   // [own][2] classes with Type I feedback
    uint32_t *type2 = type1 + 2 * own_max;                              // [own][2] classes with Type II feedback
    int32_t *octets_of = (int32_t *)(type2 + 2 * own_max);              // [own][depth] octets of a bank's list
    int32_t *incl_of = octets_of + own_max * depth;                     // [own][depth] included literals
    uint32_t *stale = (uint32_t *)(incl_of + own_max * depth);          // [own][depth] the bank's include words have changed
    int32_t *stale_list = (int32_t *)(stale + own_max * depth);         // [own * depth] ... listed
    int32_t *node_of = stale_list + own_max * depth;                    // [own] picked node, -1: none
    int32_t *learns_of = node_of + own_max;                             // [own] a node, and few enough literals (Type I in full)
    uint32_t *pick_of = (uint32_t *)(learns_of + own_max);              // [own] random word of the node pick, drawn a step ahead
    int32_t *busy_list = (int32_t *)(pick_of + own_max);                // [own] clauses that get feedback
    uint32_t *busy_of = (uint32_t *)(busy_list + own_max);              // [own] ... listed
    int32_t *own_id = (int32_t *)(busy_of + own_max);                   // [own] the clause in a slot
    uint32_t *send_row = (uint32_t *)(own_id + own_max);                // [own][NM][MB] rows that a clause sends to along a move
    uint32_t *mlit = send_row + (size_t)own_max * NM * p.MB;            // [own][MW] what the picked node received in the last layer

    if (tid == 0) {
        int n = 0;
        for (int cl = 0; cl < own_max; ++cl) {
            const int c = p.perm ? p.perm[g * own_max + cl] : (g * own_max + cl < p.C ? g * own_max + cl : -1);
            if (c >= 0) own_id[n++] = c;
        }
        n_own_shared = n, go_on = 1, n_busy = 0, n_stale = 0, next_unit = 0;
    }
    if (tid < 64) votes[tid] = 0;
    __syncthreads();
    const int n_own = __builtin_amdgcn_readfirstlane(n_own_shared);
    const int last = p.first_example + p.n_examples - 1;
    const int all_rows = p.literals + p.n_types + 1;

    auto bank_of = [&](int bank) {  // (static indices: the parameters stay in scalar registers)
        uint32_t *at = p.bank[0];
#pragma unroll
        for (int l = 1; l < GTM_MAX_DEPTH; ++l)
            if (l == bank) at = p.bank[l];
        return at;
    };
    auto threshold_of = [&](int bank) {
        uint32_t t = p.thr16[0];
#pragma unroll
        for (int l = 1; l < GTM_MAX_DEPTH; ++l)
            if (l == bank) t = p.thr16[l];
        return t;
    };
    auto planes_in_memory = [&](int c, int bank, int wl) { return bank_of(bank) + ((int64_t)c * (bank == 0 ? LA : MC) + wl) * B; };
    auto list_of = [&](int cl, int bank) {
        const int at = cl * list_entries + (bank == 0 ? 0 : p.list0 + (bank - 1) * p.listm);
        if constexpr (REGS)
            return (uint16_t *)lists_lds + at;
        else
            return p.lists + ((int64_t)g * own_max * list_entries + at);
    };
    // one wave: the list of a slot's bank from its include words, a lane per word: as many turns as the fullest word has literals
    auto make_list = [&](int cl, int bank) {
        uint16_t *list = list_of(cl, bank);
        const uint32_t *from = inc + (size_t)cl * words_all + (bank == 0 ? 0 : LA + (bank - 1) * MC);
        int n = 0, included = 0;  // n: entries so far, whole octets before the negated half
        if (bank == 0) {
            if (lane == 0) list[0] = (uint16_t)(p.literals + own_id[cl] % p.n_types);
            n = 1;
        }
        const int words = bank == 0 ? LA : MC, half = bank == 0 ? LA : MW;
        int again = bank == 0 ? p.literals + own_id[cl] % p.n_types : -1;  // an entry of the sign at hand, to fill an octet up with
        auto fill_up = [&]() {
            const int full = (n + 7) & ~7;
            if (n + lane < full) list[n + lane] = (uint16_t)again;
            n = full;
        };
        for (int w0 = 0; w0 < words;) {
            const int w1 = min(words, w0 < half ? min(half, w0 + 64) : w0 + 64);  // (a pass holds words of one sign)
            uint32_t mine = w0 + lane < w1 ? from[w0 + lane] : 0u;
            if (bank == 0 && w0 + lane == LA - 1) mine &= p.filter;
            const int first = w0 < half ? 32 * w0 : 0x8000 | (32 * (w0 - half)), own = __popc(mine), up_to = fitl_sum_up_to(own);
            const unsigned long long some = __ballot(mine != 0u);
            if (some != 0ull) {
                const int at = __ffsll((long long)some) - 1;
                if (again < 0) again = first + 32 * at + __builtin_ctz(__builtin_amdgcn_readlane(mine, at));
                uint16_t *to = list + (n + up_to - own);
                for (uint32_t m = mine; m; m &= m - 1) *to++ = (uint16_t)(first + 32 * lane + __builtin_ctz(m));
                const int more = __builtin_amdgcn_readlane(up_to, 63);
                n += more, included += more;
            }
            w0 = w1;
            if (w0 == half || w0 == words) {
                fill_up();
                again = -1;
            }
        }
        if (lane == 0) octets_of[cl * depth + bank] = n >> 3, incl_of[cl * depth + bank] = included, stale[cl * depth + bank] = 0u;
    };

    // own state -> LDS and registers
    for (int i = tid; i < n_own * words_all; i += FITP_BLOCK) {
        const int cl = i / words_all, w = i - cl * words_all;
        const int bank = w < LA ? 0 : 1 + (w - LA) / MC, wl = w < LA ? w : (w - LA) % MC;
        inc[i] = planes_in_memory(own_id[cl], bank, wl)[B - 1];
    }
    for (int i = tid; i < n_own * K; i += FITP_BLOCK) {
        const int cl = i / K, k = i - cl * K;
        wts[i] = p.weights[(int64_t)k * p.C + own_id[cl]];
    }
    for (int i = tid; i < n_own * NM * p.MB; i += FITP_BLOCK) {
        const int cl = i / (NM * p.MB), r = i - cl * NM * p.MB, k = r / p.MB, j = r - k * p.MB;
        uint32_t type = 0u;
#pragma unroll
        for (int m = 0; m < TILE_MOVES_MAX; ++m)
            if (m == k) type = (uint32_t)p.moves.type[m];
        send_row[i] = (p.hv[(int64_t)own_id[cl] * p.MB + j] + type) % (uint32_t)M;
    }
    auto draw_pick = [&](int cl, uint32_t step) {
        return philox4x32_10((uint32_t)own_id[cl], 0u, step, GTM_TAG_CLAUSE_NODE, p.k0, p.k1).v[0];
    };
    for (int cl = tid; cl < n_own; cl += FITP_BLOCK) pick_of[cl] = draw_pick(cl, p.first_step);
    int parts_log = 0;  // waves that share a clause
    while ((2 << parts_log) * own_max <= WAVES) ++parts_log;
    const int parts = 1 << parts_log, part = wave & (parts - 1);
    const int wave_cl = wave >> parts_log;  // the wave's clause, where a workgroup has at most as many clauses as waves
    // REGS: a lane keeps one automaton word of the wave's clause, or two; or four lanes keep one, each drawing a quarter of its
    // Type I bits.  What the decisions take, every wave of the clause keeps as well: lane k the weight of class k and
    // its random words, lane 63 the one of the next node pick.
    const bool owns = REGS && wave_cl < n_own;
    const int clause_lanes = 64 << parts_log, quad_log = words_all * 4 <= clause_lanes ? 2 : 0;
    const bool two_words = words_all > clause_lanes;
    struct Place {
        int w, bank, wl;
        bool there;
    };
    auto place_of = [&](int r) {
        Place at;
        at.w = (((part << 6) | lane) >> quad_log) + r * clause_lanes;
        at.there = owns && at.w < words_all;
        at.bank = 0, at.wl = at.w;
        if (at.w >= LA) {
            at.bank = 1, at.wl = at.w - LA;
            while (at.wl >= MC) at.wl -= MC, ++at.bank;
        }
        return at;
    };
    const int my_id = owns ? own_id[wave_cl] : 0;
    uint32_t planes[2][MAXB] = {};
    int32_t weight = 0;
    philox_out drawn = {};
    auto draw = [&](uint32_t step) {
        const bool pick = lane == 63;
        drawn = philox4x32_10((uint32_t)my_id, pick ? 0u : (uint32_t)lane, pick ? step + 1u : step,
                              pick ? (uint32_t)GTM_TAG_CLAUSE_NODE : (uint32_t)GTM_TAG_CLAUSE_UPDATES, p.k0, p.k1);
    };
    if (owns) {
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const Place at = place_of(r);
            if (!at.there || (r == 1 && !two_words)) continue;
            const uint32_t *from = planes_in_memory(my_id, at.bank, at.wl);
#pragma unroll
            for (int b = 0; b < MAXB; ++b)
                if (EXACT || b < B) planes[r][b] = from[b];
        }
        if (lane < K) weight = p.weights[(int64_t)lane * p.C + my_id];
        draw(p.first_step - 1u);  // (the pick of the first step)
    }
    fits_word<MAXB, EXACT> word0(planes[0], B), word1(planes[1], B);
    // the (clause, class) pair that this thread decides first (not REGS)
    const int pair_cl = tid / K, pair_k = tid - pair_cl * K;
    const uint32_t by_words = 0xFFFFFFFFu / (uint32_t)words_all;  // (a quotient from it is one too low at most)

    int n_now = (int)p.n_nodes[p.first_example], n_next = (int)p.n_nodes[min(p.first_example + 1, last)];
    uint32_t base_now = p.node_index[p.first_example], base_next = p.node_index[min(p.first_example + 1, last)];
    FitGraph fg = fit_graph_slot(p.tg, p.first_example, n_now);
    auto rows_of = [&](const FitGraph &f) { return p.tiles + (int64_t)f.tile * p.tg.rows * p.tg.tw + f.word0; };
    const uint32_t *tile_now = rows_of(fg);
    if constexpr (ROWS_LDS) {
        FitRowLoader all;
        all.prepare(fg.words, FITP_BLOCK, tid);
        all.request(tile_now, p.tg.tw, all_rows, fg.words, rows_both + wave * 64, FITP_BLOCK, tid);
    }
    for (int i = tid; i < NM * S; i += FITP_BLOCK) ends[i] = p.masks[i];
    if (tid < K) labels[0][tid] = p.encoded_Y[(int64_t)p.first_example * K + tid];
    __syncthreads();
    for (int u = wave; u < n_own * depth; u += WAVES) make_list(u / depth, u % depth);
    if (parts > 1)
        for (int i = tid; i < n_own * S; i += FITP_BLOCK) truth[i] = 0xFFFFFFFFu;
    __builtin_amdgcn_s_waitcnt(FITP_WAIT_VMEM);
    __syncthreads();

    constexpr int LOADERS = POLL * 64;  // threads that request the next graph's words
    FitRowLoader loader{};
    int loader_words = 0;
    const uint32_t *sizes = lane & 1 ? p.node_index : p.n_nodes;  // (a value per lane: nothing waits for it before it is used)
    int place = 2 * (lane & ((1 << lg) - 1));
    // Per-lane addresses are worked out anew in every phase: kept over the whole loop, as the compiler would, sixty of them were
    // spilled to memory and fetched back one by one on the step's longest path (14.1 -> 13.7 us per example on the chains).
    auto refresh = [&]() {
        asm volatile("" : "+v"(tid));
        lane = tid & 63, place = 2 * (lane & ((1 << lg) - 1));
    };
    // Words that a lane sends by one atomic.  Two where a workgroup has many clauses: on the 841-node grids, 128 rows a workgroup and
    // layer, sending took 2.9 us word by word, 2.0 in pairs.  With few (REGS) one turn of the threads sends all, and a lane is done sooner with
    // one word (1,000-node chains, 2 rows: 0.71 against 0.76 us).
    constexpr int SENT = REGS ? 1 : 2;
    int row_log = 2;  // 2^row_log lanes send a row
    while ((SENT << row_log) < S) ++row_log;
    const int by_moves = NM > 0 ? (65536 + NM - 1) / NM : 0;
    const int layer_words = M * S;
    const int share_lo = (int)((int64_t)g * layer_words / G), share_hi = (int)((int64_t)(g + 1) * layer_words / G);
    unsigned long long seen[3] = {};
    int slot = 0;

    // what a wave does with a clause on the rows of layer `bank` (0: the graph's literals); `last_layer`: node and votes as well
    auto pick_and_vote = [&](int cl, uint2 v) {
        const uint32_t random = REGS ? (uint32_t)__builtin_amdgcn_readlane(drawn.v[0], 63) : pick_of[cl];
        const int node = n_now > 0 ? fitl_pick_node(v, random, lane) : -1;
        const bool fired = n_now == 0 || node >= 0;  // (the reference's arithmetic for a graph without nodes, kernels.py:289-295)
        if (lane == 0) {
            int included = 0;
            for (int b = 0; b < depth; ++b) included += incl_of[cl * depth + b];
            node_of[cl] = node, learns_of[cl] = node >= 0 && included <= p.max_included;
        }
        if (fired && lane < K) atomicAdd(&votes[lane], REGS ? weight : wts[cl * K + lane]);
    };
    auto truth_row = [&](int cl) {
        const uint2 v = *reinterpret_cast<const uint2 *>(truth + cl * S + (place < S ? place : 0));
        return place < S ? v : make_uint2(0u, 0u);
    };
    auto evaluate = [&](int cl, int part, int bank, int i) {
        const int n8 = __builtin_amdgcn_readfirstlane(octets_of[cl * depth + bank]);
        const uint4 *list = reinterpret_cast<const uint4 *>(list_of(cl, bank));
        uint2 v;
        if (bank == 0) {
            const uint2 ones = make_uint2(0xFFFFFFFFu, 0xFFFFFFFFu);
            uint2 acc;
            if constexpr (ROWS_LDS) {
                const int stride = fitl_stride(fg.words);
                acc = fitm_rows<false, uint2>(ones, list, n8, part, parts, rows_both + (i & 1) * p.rows_words + (place < stride ? place : 0),
                                              stride, lg, lane);
            } else {
                acc = fitm_rows<false, fitm_pair>(ones, list, n8, part, parts, tile_now + (place < fg.words ? place : 0), p.tg.tw, lg, lane);
            }
            v = fitl_nodes(make_uint2(fitl_and_groups(acc.x, lg), fitl_and_groups(acc.y, lg)), fg, lg, lane);
        } else {
            const uint2 before = truth_row(cl);
            v = before;
            if (__ballot((before.x | before.y) != 0u) != 0ull) {
                const uint2 acc = fitm_rows<true, uint2>(before, list, n8, part, parts, mrows + (place < S ? place : 0), S, lg, lane);
                v = make_uint2(fitl_and_groups(acc.x, lg), fitl_and_groups(acc.y, lg));
            }
            if (lane >= (1 << lg)) v = make_uint2(0u, 0u);
        }
        if (lane < (S >> 1)) {
            if (parts == 1)
                *reinterpret_cast<uint2 *>(truth + cl * S + 2 * lane) = v;
            else
                atomicAnd(&truth[cl * S + 2 * lane], v.x), atomicAnd(&truth[cl * S + 2 * lane + 1], v.y);
        }
        if (parts == 1 && bank == L) pick_and_vote(cl, v);
    };
    auto evaluate_all = [&](int bank, int i) {
        if (own_max <= WAVES) {
            if (wave_cl < n_own) evaluate(wave_cl, part, bank, i);
        } else {  // (clauses differ a lot in what they cost: the waves take them from a queue)
            for (;;) {
                int u = 0;
                if (lane == 0) u = atomicAdd(&next_unit, 1);
                u = __builtin_amdgcn_readfirstlane(u);
                if (u >= n_own) break;
                evaluate(u, 0, bank, i);
            }
        }
    };

    for (int i = 0; i < p.n_examples; ++i) {
        const uint32_t step = p.first_step + (uint32_t)i;
        const int ex = p.first_example + i;
        refresh();
        uint32_t *got_now = p.got + (size_t)slot * L * layer_words, *got_next = p.got + (size_t)(slot == 2 ? 0 : slot + 1) * L * layer_words;
        // ---- 1. layer 0 (K1)
        evaluate_all(0, i);
        FitGraph fn = fg;
        uint32_t after = 0u;
        bool alive = true;

        // ---- 2. the message layers
        for (int l = 0; l < L; ++l) {
            lds_barrier();  // the truth rows are complete, and nobody reads the received rows of the layer before
            refresh();
            uint32_t *got_l = got_now + (size_t)l * layer_words;
            if (tid == 0) next_unit = 0, next_words = 0;
            if constexpr (COLLECT) {  // (the rows received before are not read any more)
                for (int at = tid; at < layer_words / 2; at += FITP_BLOCK) ((unsigned long long *)mrows)[at] = 0ull;
                lds_barrier();
                refresh();
            }
            // a. what the own clauses make the nodes receive: their truth rows, shifted, where an edge of the move ends
            for (int u = tid >> row_log; u < n_own * NM; u += FITP_BLOCK >> row_log) {
                const int cl = (u * by_moves) >> 16, k = u - cl * NM, w = SENT * (tid & ((1 << row_log) - 1));
                int shift_words = 0, shift_bits = 0;
#pragma unroll
                for (int m = 0; m < TILE_MOVES_MAX; ++m)
                    if (m == k) shift_words = p.moves.words[m], shift_bits = p.moves.bits[m];
                const uint32_t *row = truth + cl * S;
                auto word = [&](int q) { return q >= 0 && q < S ? row[q] : 0u; };
                const uint32_t *to = ends + ((i & 1) * NM + k) * S + w;
                const uint32_t t0 = word(w + shift_words), t1 = word(w + shift_words + 1);
                uint64_t v = w < fg.words ? __builtin_amdgcn_alignbit(t1, t0, shift_bits) & to[0] : 0u;
                if (SENT == 2 && w + 1 < fg.words)  // (S is even)
                    v |= (uint64_t)(__builtin_amdgcn_alignbit(word(w + shift_words + 2), t1, shift_bits) & to[SENT - 1]) << 32;
                if (v != 0u)
                    for (int j = 0; j < p.MB; ++j) {
                        uint32_t *at = got_l + send_row[u * p.MB + j] * (uint32_t)S + w;
                        if constexpr (COLLECT)
                            atomicOr((unsigned long long *)(mrows + (at - got_l)), (unsigned long long)v);
                        else if constexpr (SENT == 2)
                            __hip_atomic_fetch_or((unsigned long long *)at, (unsigned long long)v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        else
                            __hip_atomic_fetch_or(at, (uint32_t)v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    }
            }
            if constexpr (COLLECT) {
                lds_barrier();
                refresh();
                for (int at = tid; at < layer_words / 2; at += FITP_BLOCK) {
                    const unsigned long long v = ((const unsigned long long *)mrows)[at];
                    if (v != 0ull) __hip_atomic_fetch_or((unsigned long long *)got_l + at, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
            __builtin_amdgcn_s_waitcnt(FITP_WAIT_VMEM);  // the ORs have been carried out where every workgroup sees them
            asm volatile("" ::: "memory");
            lds_barrier();
            refresh();
            unsigned long long *arrived = p.arrived + (size_t)l * FITD_PARTS * FITD_STRIDE;
            if (wave == POLL) {
                if (lane == 0)
                    __hip_atomic_fetch_add(&arrived[(g % FITD_PARTS) * FITD_STRIDE], 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                const unsigned long long everyone = (unsigned long long)(i + 1) * (unsigned long long)G;
                uint32_t polls = 0;
                unsigned long long waiting_since = 0ull;
                bool ok = !p.force_abort;
                if (!ok) __hip_atomic_store(p.abort_flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                while (ok) {  // (the abort flag travels with the counters)
                    int v = (int)(uint32_t)__hip_atomic_load(&arrived[lane * FITD_STRIDE], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    const uint32_t aborted = __builtin_amdgcn_readfirstlane(__hip_atomic_load(p.abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
                    v = __builtin_amdgcn_readlane(fitl_sum_up_to(v), 63);
                    if ((uint32_t)v >= (uint32_t)everyone) break;
                    if (aborted != 0 || fit_wait_is_over(polls, p.spin_limit, waiting_since, p.wait_ticks)) {
                        __hip_atomic_store(p.abort_flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        ok = false;
                    }
                }
                if (!ok && lane == 0) go_on = 0;
            } else {
                // (meanwhile) this group's share of the slot that the next example will send into; the next graph's words
                for (int at = share_lo + tid; at < share_hi; at += LOADERS)
                    __hip_atomic_store(&got_next[(size_t)l * layer_words + at], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (l == 0 && i + 1 < p.n_examples) {
                    const FitGraph next = fit_graph_slot(p.tg, ex + 1, n_next);
                    if constexpr (ROWS_LDS) {
                        if (next.words != loader_words) loader_words = next.words, loader.prepare(next.words, LOADERS, tid);
                        loader.request(rows_of(next), p.tg.tw, all_rows, next.words, rows_both + (~i & 1) * p.rows_words + wave * 64, LOADERS, tid);
                    }
                    const uint32_t *from = p.masks + (int64_t)(i + 1) * NM * S;
                    uint32_t *to = ends + (~i & 1) * NM * S + wave * 64;
                    for (int at = 0; at < NM * S; at += LOADERS)
                        if (at + tid < NM * S) fitp_load_to_lds(from + at + tid, to + at);
                    if (wave == POLL - 1 && lane < K)
                        fitp_load_to_lds((const uint32_t *)p.encoded_Y + (int64_t)(ex + 1) * K + lane, (uint32_t *)labels[~i & 1]);
                }
            }
            __builtin_amdgcn_s_waitcnt(FITP_WAIT_VMEM);
            lds_barrier();
            if (!go_on) {
                alive = false;
                break;
            }
            // b. the received rows -> LDS
            refresh();
            {
                const unsigned long long *from = (const unsigned long long *)got_l;
                unsigned long long *to = (unsigned long long *)mrows;
                const int pairs = layer_words / 2;
                for (int at0 = tid; at0 < pairs; at0 += 8 * FITP_BLOCK) {
                    unsigned long long v[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u)
                        v[u] = at0 + u * FITP_BLOCK < pairs ? __hip_atomic_load(&from[at0 + u * FITP_BLOCK], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                                                            : 0ull;
#pragma unroll
                    for (int u = 0; u < 8; ++u)
                        if (at0 + u * FITP_BLOCK < pairs) to[at0 + u * FITP_BLOCK] = v[u];
                }
            }
            lds_barrier();
            refresh();
            // c. K2 for the own clauses; what the nodes of this group's share received, node-major, for the feedback
            evaluate_all(l + 1, i);
            if (l < L - 1) {
                const int v_lo = (int)((int64_t)g * n_now / G), v_hi = (int)((int64_t)(g + 1) * n_now / G);
                uint32_t *vec_l = p.vec + (size_t)l * p.max_nodes * MW;
                for (int j = wave; 64 * j < M; j += WAVES)
                    for (int v = v_lo; v < v_hi; ++v) {
                        const int r = 64 * j + lane;
                        const unsigned long long got = __ballot(r < M && ((mrows[r * S + (v >> 5)] >> (v & 31)) & 1u));
                        if (lane < 2 && 2 * j + lane < MW)
                            __hip_atomic_store(&vec_l[(size_t)v * MW + 2 * j + lane], (uint32_t)(got >> (32 * lane)), __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT);
                    }
            }
        }
        if (!alive) break;
        if (parts > 1) {  // ---- 3. node pick (K7) and votes (K6) of clauses that several waves share
            lds_barrier();
            if (part == 0 && wave_cl < n_own) {
                const uint2 v = truth_row(wave_cl);
                pick_and_vote(wave_cl, lane < (1 << lg) ? v : make_uint2(0u, 0u));
            }
        }
        // the next slot's share is cleared (and the node-major words are out) before this group arrives
        __builtin_amdgcn_s_waitcnt(FITP_WAIT_VMEM);
        asm volatile("" ::: "memory");
        lds_barrier();

        // ---- 4. class sums across the device (the protocol of fit_persistent.h); meanwhile all that does not need them
        refresh();
        unsigned long long *slot_sum = p.class_sum + (size_t)slot * K * FITP_SUM_PARTS * FITP_SUM_STRIDE;
        if (wave == POLL) {
            if (lane < K) {
                __hip_atomic_fetch_add(&slot_sum[(lane * FITP_SUM_PARTS + g % FITP_SUM_PARTS) * FITP_SUM_STRIDE],
                                       FITP_ARRIVED + (unsigned long long)(long long)votes[lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                votes[lane] = 0;
            }
        } else {
            // what the picked nodes received in the last layer: 64 rows at a time, a ballot of the node's bits
            const int pairs_of_words = (M + 63) >> 6;
            for (int u = wave; u < n_own * pairs_of_words; u += POLL) {
                const int cl = u / pairs_of_words, j = u - cl * pairs_of_words;
                const int node = __builtin_amdgcn_readfirstlane(node_of[cl]);
                if (node < 0) continue;
                const int r = 64 * j + lane;
                const unsigned long long got = __ballot(r < M && ((mrows[r * S + (node >> 5)] >> (node & 31)) & 1u));
                if (lane < 2 && 2 * j + lane < MW) mlit[cl * MW + 2 * j + lane] = (uint32_t)(got >> (32 * lane));
            }
            if (parts > 1)
                for (int at = tid; at < n_own * S; at += LOADERS) truth[at] = 0xFFFFFFFFu;
            if (tid == 0) n_busy = 0, n_stale = 0, next_unit = 0;
            if constexpr (!REGS)
                for (int at = tid; at < 2 * n_own; at += LOADERS) type1[at] = 0u, type2[at] = 0u, busy_of[at >> 1] = 0u;
            for (int j = tid; !REGS && j < n_own * (K + 1); j += LOADERS) {
                if (j >= n_own * K) {
                    pick_of[j - n_own * K] = draw_pick(j - n_own * K, step + 1u);
                    continue;
                }
                const int cl = j == tid ? pair_cl : j / K, k = j - cl * K;
                const philox_out r = philox4x32_10((uint32_t)own_id[cl], (uint32_t)k, step, GTM_TAG_CLAUSE_UPDATES, p.k0, p.k1);
                gate[2 * j] = r.v[0], gate[2 * j + 1] = r.v[1];
            }
        }
        uint32_t x0 = 0u, x1 = 0u;  // REGS: the literal words of the picked node for this lane's words
        if constexpr (REGS) {
            if (owns) {
                const int node = __builtin_amdgcn_readfirstlane(node_of[wave_cl]);
                if (node >= 0) {
                    const uint32_t *from = p.X + ((int64_t)base_now + node) * LA;
                    const int w = ((part << 6) | lane) >> quad_log;
                    if (w < LA) x0 = from[w];
                    if (w + clause_lanes < LA) x1 = from[w + clause_lanes];
                }
                draw(step);
            }
        }
        fn = fit_graph_slot(p.tg, min(ex + 1, last), n_next);
        after = sizes[min(ex + 2, last)];
        if (wave == POLL && lane < K) {
            const unsigned long long everyone = (unsigned long long)G;
            uint32_t polls = 0;
            unsigned long long waiting_since = 0ull, sum = 0ull;
            bool ok = !p.force_abort;
            if (!ok) __hip_atomic_store(p.abort_flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            while (ok) {
                unsigned long long part[FITP_SUM_PARTS];
#pragma unroll
                for (int s = 0; s < FITP_SUM_PARTS; ++s)
                    part[s] = __hip_atomic_load(&slot_sum[(lane * FITP_SUM_PARTS + s) * FITP_SUM_STRIDE], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                const uint32_t aborted = __hip_atomic_load(p.abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                sum = 0ull;
#pragma unroll
                for (int s = 0; s < FITP_SUM_PARTS; ++s) sum += part[s];
                if ((((sum - seen[0] + FITP_HALF) >> 48) & 0xFFFFull) == everyone) break;
                if (aborted != 0 || fit_wait_is_over(polls, p.spin_limit, waiting_since, p.wait_ticks)) {
                    __hip_atomic_store(p.abort_flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    ok = false;
                    break;
                }
            }
            if (!ok) go_on = 0;
            sums[lane] = (int32_t)(long long)(sum - seen[0] - (everyone << 48));
            seen[0] = seen[1], seen[1] = seen[2], seen[2] = sum;
        }
        __builtin_amdgcn_s_waitcnt(FITP_WAIT_VMEM);
        lds_barrier();
        if (!go_on) break;

        // ---- 5. feedback decisions (K8) and weights
        refresh();
        auto decide = [&](int k, int32_t &w, uint32_t r0, uint32_t r1, bool fired) {
            int cs = sums[k];
            cs = cs > p.T ? p.T : (cs < -p.T ? -p.T : cs);
            const int y = labels[i & 1][k];
            const int target = 1 - 2 * (cs > y);
            const int sign = w >= 0 ? 1 : -1;
            int err = y - cs;
            err = err < 0 ? -err : err;
            const bool skip = (target == -1 && (uint64_t)r0 >= p.q_thr) || ((uint64_t)r1 * (uint64_t)(2 * (int64_t)p.T) >= ((uint64_t)err << 32));
            const int u = skip ? 0 : target * sign;
            if (u > 0 && fired && (w < 0 ? -(int64_t)w : (int64_t)w) < 2147483647) {
                w += sign;
            } else if (u < 0 && fired) {
                w -= sign;
                if (p.negative == 0 && w < 1) w = 1;
            }
            return u;
        };
        if constexpr (!REGS) {
            for (int j = tid; j < n_own * K; j += FITP_BLOCK) {
                const int cl = j == tid ? pair_cl : j / K, k = j == tid ? pair_k : j - cl * K;
                int32_t w = wts[j];
                const int u = decide(k, w, gate[2 * j], gate[2 * j + 1], node_of[cl] >= 0);
                if (u == 0) continue;
                wts[j] = w;
                atomicOr(&type1[(u > 0 ? 0 : 2 * own_max) + 2 * cl + (k >> 5)], 1u << (k & 31));
                if (atomicOr(&busy_of[cl], 1u) == 0u) busy_list[atomicAdd(&n_busy, 1)] = cl;
            }
            lds_barrier();
        }

        // ---- 6. Type I / II feedback on every bank (K9, K10)
        refresh();
        // the literal word of a clause's picked node (kernels.py:592-615: the negated half of a message is the complement)
        auto message_word = [&](int cl, int node, int bank, int wl) {
            const int w = wl < MW ? wl : wl - MW;
            uint32_t v;
            if (bank == L)
                v = mlit[cl * MW + w];
            else
                v = fitd_load(&p.vec[((size_t)(bank - 1) * p.max_nodes + node) * MW + w]);
            return wl < MW ? v : ~v;
        };
        if constexpr (REGS) {
            if (owns) {
                const int node = __builtin_amdgcn_readfirstlane(node_of[wave_cl]);
                const bool fired = node >= 0;
                const int u = lane < K ? decide(lane, weight, drawn.v[0], drawn.v[1], fired) : 0;
                const unsigned long long pos = __ballot(u > 0), neg = __ballot(u < 0);
                if ((pos | neg) != 0ull) {
                    const bool learns = __builtin_amdgcn_readfirstlane(learns_of[wave_cl]) != 0;
                    const Place at0 = place_of(0);
                    if (fired && at0.there && at0.bank != 0) x0 = message_word(wave_cl, node, at0.bank, at0.wl);
                    const uint32_t was0 = word0.top();
                    auto update = [&](fits_word<MAXB, EXACT> &word, const Place &at, uint32_t x, uint32_t threshold) {
                        for (unsigned long long m = pos | neg; m != 0ull; m &= m - 1) {
                            const int k = __ffsll((long long)m) - 1;
                            uint32_t up = fired ? ~x & ~word.top() : 0u, down = 0u;
                            if ((pos >> k) & 1ull) {
                                uint32_t fb;
                                if (quad_log == 2) {
                                    fb = fitl_feedback_byte(p.k0, p.k1, (uint32_t)my_id, (uint32_t)at.wl, (uint32_t)lane & 3u, step, (uint32_t)at.bank,
                                                            (uint32_t)k, threshold)
                                         << (8 * (lane & 3));
                                    fb |= (uint32_t)__builtin_amdgcn_mov_dpp((int)fb, 0xB1, 0xF, 0xF, true);  // lanes of a quad: [1, 0, 3, 2]
                                    fb |= (uint32_t)__builtin_amdgcn_mov_dpp((int)fb, 0x4E, 0xF, 0xF, true);  // [2, 3, 0, 1]
                                } else {
                                    fb = gtm_feedback_bits(p.k0, p.k1, (uint32_t)my_id, (uint32_t)at.wl, step, (uint32_t)at.bank, (uint32_t)k, threshold);
                                }
                                up = learns ? (p.boost == 1 ? x : x & ~fb) : 0u;
                                down = learns ? ~x & fb : fb;
                            }
                            word.count(up, down);
                        }
                    };
                    auto note = [&](const Place &at, uint32_t top) {
                        inc[wave_cl * words_all + at.w] = top;
                        stale[wave_cl * depth + at.bank] = 1u;
                        n_stale = 1;
                    };
                    if (at0.there) {
                        update(word0, at0, x0, threshold_of(at0.bank));
                        if (word0.top() != was0) note(at0, word0.top());
                    }
                    if (two_words) {
                        const Place at1 = place_of(1);
                        if (at1.there) {
                            if (fired && at1.bank != 0) x1 = message_word(wave_cl, node, at1.bank, at1.wl);
                            const uint32_t was1 = word1.top();
                            update(word1, at1, x1, threshold_of(at1.bank));
                            if (word1.top() != was1) note(at1, word1.top());
                        }
                    }
                }
            }
            lds_barrier();
            if (n_stale != 0) {
                for (int bank = part; owns && bank < depth; bank += parts)
                    if (__builtin_amdgcn_readfirstlane(stale[wave_cl * depth + bank]) != 0u) make_list(wave_cl, bank);
                lds_barrier();
            }
        } else {
            // the words of the clauses that get feedback, shared out; a thread's next word is fetched while it works on one
            struct Fetched {
                uint32_t planes[MAXB], x;
                int cl, bank, wl, w;
            };
            auto fetch = [&](Fetched &f, int b, int w) {
                f.cl = busy_list[b], f.w = w, f.bank = 0, f.wl = w;
                if (w >= LA) {
                    f.bank = 1, f.wl = w - LA;
                    while (f.wl >= MC) f.wl -= MC, ++f.bank;
                }
                const uint32_t *from = planes_in_memory(own_id[f.cl], f.bank, f.wl);
                if (EXACT && MAXB == 8 && ((uintptr_t)from & 15u) == 0) {
                    const uint4 lo = reinterpret_cast<const uint4 *>(from)[0], hi = reinterpret_cast<const uint4 *>(from)[1];
                    f.planes[0] = lo.x, f.planes[1] = lo.y, f.planes[2] = lo.z, f.planes[3] = lo.w;
                    f.planes[4 % MAXB] = hi.x, f.planes[5 % MAXB] = hi.y, f.planes[6 % MAXB] = hi.z, f.planes[7 % MAXB] = hi.w;
                } else {
#pragma unroll
                    for (int q = 0; q < MAXB; ++q) f.planes[q] = EXACT || q < B ? from[q] : 0u;
                }
                const int node = node_of[f.cl];
                f.x = 0u;
                if (node >= 0) {
                    if (f.bank == 0)
                        f.x = p.X[((int64_t)base_now + node) * LA + f.wl];
                    else
                        f.x = message_word(f.cl, node, f.bank, f.wl);
                }
            };
            // 64 words at a time off a queue: what a word costs depends on its clause's feedback (in turns of all threads 15.6 us
            // on the 841-node grids, the last of five turns nearly empty; 14.5 off the queue)
            const int total = n_busy * words_all;
            auto take = [&](Fetched &f) {
                int at = 0;
                if (lane == 0) at = atomicAdd(&next_words, 64);
                at = __builtin_amdgcn_readfirstlane(at) + lane;
                f.cl = -1;
                if (at < total) {
                    int b = (int)__umulhi((uint32_t)at, by_words), w = at - b * words_all;
                    if (w >= words_all) w -= words_all, ++b;
                    fetch(f, b, w);
                }
                return at - lane < total;
            };
            Fetched now, next;
            for (bool more = take(now); more; now = next) {
                more = take(next);
                if (now.cl < 0) continue;
                fits_word<MAXB, EXACT> state(now.planes, B);
                const uint32_t was = state.top(), c = (uint32_t)own_id[now.cl];
                const bool fired = node_of[now.cl] >= 0, learns = learns_of[now.cl] != 0;
                const uint32_t threshold = threshold_of(now.bank), x = now.x;
                for (int h = 0; h < 2; ++h) {
                    const uint32_t pos = type1[2 * now.cl + h];
                    for (uint32_t m = pos | type2[2 * now.cl + h]; m; m &= m - 1) {
                        const int k = __builtin_ctz(m);
                        uint32_t up = fired ? ~x & ~state.top() : 0u, down = 0u;
                        if ((pos >> k) & 1u) {
                            const uint32_t fb = gtm_feedback_bits(p.k0, p.k1, c, (uint32_t)now.wl, step, (uint32_t)now.bank, (uint32_t)(32 * h + k), threshold);
                            up = learns ? (p.boost == 1 ? x : x & ~fb) : 0u;
                            down = learns ? ~x & fb : fb;
                        }
                        state.count(up, down);
                    }
                }
                state.store(planes_in_memory(own_id[now.cl], now.bank, now.wl));
                if (state.top() != was) {
                    inc[now.cl * words_all + now.w] = state.top();
                    if (atomicOr(&stale[now.cl * depth + now.bank], 1u) == 0u) stale_list[atomicAdd(&n_stale, 1)] = now.cl * depth + now.bank;
                }
            }
            __syncthreads();
            refresh();
            const int n_changed = n_stale;
            if (n_changed != 0) {
                for (int u = wave; u < n_changed; u += WAVES) make_list(stale_list[u] / depth, stale_list[u] % depth);
                __syncthreads();
            }
        }
        slot = slot == 2 ? 0 : slot + 1;
        fg = fn;
        tile_now = rows_of(fg);
        n_now = n_next, base_now = base_next;
        n_next = __builtin_amdgcn_readlane(after, 0), base_next = (uint32_t)__builtin_amdgcn_readlane(after, 1);
    }
    __builtin_amdgcn_s_waitcnt(FITP_WAIT_VMEM);  // no load into LDS is left in flight when the group ends
    lds_barrier();
    // own state -> global memory (also after an abort: the host puts the model back as it was)
    if constexpr (REGS) {
        if (owns) {
            const Place at0 = place_of(0), at1 = place_of(1);
            if (at0.there && (lane & ((1 << quad_log) - 1)) == 0) word0.store(planes_in_memory(my_id, at0.bank, at0.wl));
            if (two_words && at1.there) word1.store(planes_in_memory(my_id, at1.bank, at1.wl));
            if (part == 0 && lane < K) p.weights[(int64_t)lane * p.C + my_id] = weight;
        }
    } else {
        for (int i = tid; i < n_own * K; i += FITP_BLOCK) {
            const int cl = i / K, k = i - cl * K;
            p.weights[(int64_t)k * p.C + own_id[cl]] = wts[i];
        }
    }
}
