// A whole run of training examples (the loop at tm.py:669-747) of a depth-1
// model in ONE cooperative launch.
//
// Each workgroup owns a contiguous range of clauses for the whole run and keeps
// their automata (all bit planes) and weights in LDS; they go back to global
// memory once, at the end.  (Small clauses: fit_waves.h.)  Per example a workgroup
//   1. evaluates its clauses on the graph's literal-major rows (staged in LDS;
//      the next graph's rows and labels are loaded straight into the other LDS
//      buffers while waiting at the barrier) by the clauses' lists of rows
//      (fit_lists.h), picks the nodes, and adds its clauses' votes to the class
//      sums in global memory;
//   2. meets the other workgroups at a device-wide barrier (the class sums are
//      the only thing that crosses clause boundaries, kernels.py:310-315);
//   3. decides the feedback and updates its automata and weights in LDS: the
//      (clause, class) pairs that need Type I bits and the clauses that get any
//      feedback are listed, so that every thread has a byte to draw or a word to update.
// Single-node images of 128 literal words, 2,500 clauses: 14.4 us per example with every (clause, word) looking at all
// its classes and a word's four generator calls in one thread; now 10.5.
// Class sums and barrier are one thing: class k has a 64-bit word (kept as
// FITP_SUM_PARTS partial words that a reader adds up, since the memory system
// carries out the adds to one word one after the other) to which every
// workgroup adds (1 << 48) + its share with one device-scope atomic, and which it
// then polls.  Nothing else is ever done to the word - no reset, no store - so
// per-location coherence is all the protocol needs: nothing has to be ordered
// against a separate barrier word and no cache is flushed or invalidated.  What an
// example contributed is the word now minus the word as it stood when its last use
// was complete (each polling thread remembers that value): modulo 2^64 that
// difference is arrivals * 2^48 + sum, whatever borrows negative shares caused, so
// with |sum| < 2^47 the arrivals are (difference + 2^47) >> 48 and, once they equal
// the number of workgroups, the sum is the rest.  The words live in a ring of three
// slots, each partial word in a cache line of its own (the adds and polls go to
// different memory channels): a workgroup can be one example ahead of the
// slowest one, never three.  Thread k of a workgroup polls the word of class k.
// The workgroup's barriers order LDS traffic only, so none of them waits for the
// adds or for the loads of the next graph.
//
// The wait is bounded (a few seconds of the device's wall clock; a number of polls
// in tests): a workgroup whose wait runs out raises the abort flag and every
// workgroup leaves the loop at its next check, so the grid always drains.  The
// host then puts the model back as it was and trains the examples by launches per
// example instead.
#pragma once

constexpr int FITP_BLOCK = 1024;  // 16 waves: one clause per wave in flight, four waves per SIMD hide each other's latencies

// A device-wide wait gives up after `spin_limit` polls or `wait_ticks` ticks of the wall clock (constant
// rate, whatever the shader clock does), whichever comes first.  The clock is a memory instruction of its
// own, so it is only looked at every 256th poll: an ordinary wait (a few polls) never reads it.
__device__ __forceinline__ bool fit_wait_is_over(uint32_t &polls, uint32_t spin_limit, unsigned long long &since,
                                                 unsigned long long wait_ticks) {
    if (++polls > spin_limit) return true;
    if ((polls & 255u) == 0u) {
        const unsigned long long now = wall_clock64();
        if (since == 0ull)
            since = now;
        else if (now - since > wait_ticks)
            return true;
    }
    return false;
}

struct FitPersistParams {
    // data set
    const uint32_t *tiles;
    const uint32_t *X;
    const uint32_t *node_index;
    const uint32_t *n_nodes;
    const int32_t *encoded_Y;
    TileGeom tg;
    int first_example, n_examples;
    uint32_t first_step;
    // model
    uint32_t *bank;
    int32_t *weights;
    int literals, n_types, C, LA, B, K, T, negative, boost, max_included;
    uint32_t filter, thr16, k0, k1;
    uint64_t q_thr;
    // coordination
    unsigned long long *class_sum;  // [3][K][FITP_SUM_PARTS] words FITP_SUM_STRIDE apart, zero on entry (K <= FITP_BLOCK)
    uint32_t *abort_flag;           // [1], zero on entry
    uint32_t spin_limit;  // polls after which a wait gives up (tests; 2^32 - 1 otherwise: the clock bounds the wait)
    unsigned long long wait_ticks;  // ticks of the device's wall clock after which a wait gives up
    int force_abort;      // give up at the first wait without looking (exercises the drain path)
    int clauses_per_group;
    int rows_words;       // LDS words of one staged graph: (literals + n_types + 1) * max slot words
    int max_words;        // words per graph slot that can hold nodes
    int x_words;          // LDS words of one graph's node-major literal words: max nodes * LA (DIRECT, else 0)
    const uint32_t *node_type;  // [total nodes]
    int lanes_log;        // log2 of the lanes that a row takes (fit_lists.h)
    int lists;            // entries of a clause's list of rows
    int ahead;            // the picked nodes' literal words have a place in LDS
};

constexpr unsigned long long FITP_HALF = 1ull << 47;      // class sums are smaller than this in magnitude
constexpr unsigned long long FITP_ARRIVED = 1ull << 48;   // one arrival in bits 48..63
constexpr int FITP_SUM_STRIDE = 16;                      // 64-bit words between two class-sum words (one per 128-byte line)
// A class sum is kept as this many partial words; group g adds to part g % FITP_SUM_PARTS and the
// reader adds the parts up (the protocol is linear in the word). Adds to one word are carried out
// one after the other by the memory system, so fewer groups per word shorten the exchange.
constexpr int FITP_SUM_PARTS = 16;
constexpr int FITP_DIRECT_NODES = 32;  // a node of a directly tested graph is a bit of a word

// One 32-bit word per lane from global memory straight into LDS (no register holds it meanwhile):
// lane l's word lands at dst_of_wave[l]; dst_of_wave must be the same for the whole wave. The words
// are there once the wave has waited for its vector-memory counter (FITP_WAIT_VMEM) and, for other
// waves, after the barrier that follows.
__device__ __forceinline__ void fitp_load_to_lds(const uint32_t *src, uint32_t *dst_of_wave) {
    __builtin_amdgcn_global_load_lds(src, (__attribute__((address_space(3))) uint32_t *)dst_of_wave, 4, 0, 0);
}
// Between LDS writes of some lanes of a wave and reads of them by other lanes of the same wave (the
// hardware carries out a wave's LDS accesses in order; this keeps the compiler from reordering them).
__device__ __forceinline__ void fitp_wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}
constexpr int FITP_WAIT_VMEM = 0x0F70;  // s_waitcnt vmcnt(0) (export and LDS counters left alone)


// The rows of a graph's slot -> LDS, fitl_stride(words) words apart, straight from memory (no register holds them meanwhile; they are
// there once the wave has waited for its vector-memory counter and, for other waves, after the barrier that follows).
// Threads tid < loaders (a multiple of 64) take part.
struct FitRowLoader {
    int stride, dr, dw, r0, w0;  // a thread's elements are `loaders` apart: (row, word) advance without dividing
    __device__ __forceinline__ void prepare(int words, int loaders, int tid) {
        stride = fitl_stride(words);
        dr = loaders / stride, dw = loaders - dr * stride;
        r0 = tid / stride, w0 = tid - r0 * stride;
    }
    __device__ __forceinline__ void request(const uint32_t *tile, int tw, int rows, int words, uint32_t *dst_of_wave, int loaders, int tid) const {
        if (tid >= loaders) return;
        const int total = rows * stride;
        int w = w0, row = r0 * tw;
        for (int at = 0; at < total; at += loaders) {
            if (at + tid < total) fitp_load_to_lds(tile + (row + (w < words ? w : 0)), dst_of_wave + at);
            w += dw, row += dr * tw;
            if (w >= stride) w -= stride, row += tw;
        }
    }
};

// LDS words of the kernel: `lists` = room for the clauses' lists of rows (entries per clause, a whole number of batches, 0 without),
// `ahead` = room for the literal words of the nodes that the clauses learn from.
inline size_t fit_persistent_lds_words(int per_group, int LA, int B, int K, int rows_words, int x_words, int lists, bool ahead) {
    const size_t own = (size_t)per_group, KW = (size_t)(K + 31) / 32;
    return (own * LA * B + 7) / 8 * 8 + (own * lists / 2 + 3) / 4 * 4 + 2 * (size_t)rows_words + own * K + 5 * own + 2 * (size_t)K + 2 * own * K +
           own * LA * K + own * K + 2 * own * KW + 2 * (size_t)x_words + (ahead ? own * LA : 0) + 8 * (size_t)K;
}

// MAXB: bit planes of an automaton the kernel keeps in registers while updating a word (>= B; EXACT: B itself).
// DIRECT: graphs of at most FITP_DIRECT_NODES nodes: every node is tested on its own literal words, no rows are staged.
template <int MAXB, bool EXACT, bool DIRECT>
__global__ __launch_bounds__(FITP_BLOCK) void k_fit_persistent(FitPersistParams p) {
    extern __shared__ __align__(16) uint32_t lds[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr int WAVES = FITP_BLOCK / 64;
    const int c0 = blockIdx.x * p.clauses_per_group;
    const int n_own = min(p.clauses_per_group, p.C - c0);
    const int LA = p.LA, B = EXACT ? MAXB : p.B, K = p.K, KW = (K + 31) / 32;
    const int own_max = p.clauses_per_group;

    // LDS carve-up
    uint32_t *ta = lds;                                               // [own][LA][B]
    uint16_t *lists = (uint16_t *)(ta + ((size_t)own_max * LA * B + 7) / 8 * 8);  // [own][p.lists] rows that a clause ANDs
    // (buffers of this and the next example: addressed from the first one, a choice between two pointers would make the
    // reads flat ones)
    uint32_t *rows_both = (uint32_t *)lists + ((size_t)own_max * p.lists / 2 + 3) / 4 * 4;  // [2][p.rows_words] literal-major rows
    int32_t *wts = (int32_t *)(rows_both + 2 * p.rows_words);  // [own][K]
    int32_t *node_of = wts + (size_t)own_max * K;              // [own]
    int32_t *incl_of = node_of + own_max;                      // [own] included literals
    uint32_t *stale = (uint32_t *)(incl_of + own_max);         // [own] bit 0: the include plane has changed since list and count were made; bit 1: on the busy list
    uint32_t *pick_of = stale + own_max;                       // [own] random word of the node pick, drawn a step ahead
    int32_t *busy_list = (int32_t *)(pick_of + own_max);       // [own] clauses with feedback
    int32_t *sums = busy_list + own_max;                       // [K] class sums of the example
    int32_t *votes = sums + K;                                 // [K] this group's share of the class sums
    uint32_t *gate = (uint32_t *)(votes + K);                  // [own][K][2] random words of the feedback gates
    uint32_t *fbits = gate + 2 * (size_t)own_max * K;          // [own][LA][K] Type I feedback bits
    int32_t *pair_list = (int32_t *)(fbits + (size_t)own_max * LA * K);  // [own * K] (clause, class) pairs with Type I feedback
    uint32_t *pos_of = (uint32_t *)(pair_list + (size_t)own_max * K);    // [own][KW] classes with Type I feedback
    uint32_t *neg_of = pos_of + (size_t)own_max * KW;                    // [own][KW] classes with Type II feedback
    uint32_t *x_both = neg_of + (size_t)own_max * KW;          // DIRECT: [2][nodes][LA] literal words of the graph
    uint32_t *x_ahead = x_both + 2 * p.x_words;                // [own][LA] literal words of the picked nodes (p.ahead)
    // thread k < K: its class-sum word as it stood when each of the three
    // slots was last complete (all zero before the first use): [slot][low, high][K]
    uint32_t *seen = x_ahead + (p.ahead ? (size_t)own_max * LA : 0);
    uint32_t *y_both = seen + 6 * K;                          // [2][K] labels
    __shared__ int go_on, n_pairs, n_busy;
    __shared__ uint32_t after_lds[2];
    __shared__ uint32_t types_lds[2][FITP_DIRECT_NODES];  // node types of this and the next graph (direct evaluation)

    auto draw_pick = [&](int cl, uint32_t step) {
        return philox4x32_10((uint32_t)(c0 + cl), 0u, step, GTM_TAG_CLAUSE_NODE, p.k0, p.k1).v[0];
    };

    // own state -> LDS
    for (int k = tid; k < K; k += FITP_BLOCK) votes[k] = 0;
    for (int i = tid; i < n_own * LA * B; i += FITP_BLOCK) ta[i] = p.bank[(int64_t)c0 * LA * B + i];
    for (int i = tid; i < n_own * K; i += FITP_BLOCK) {
        int cl = i / K, k = i - cl * K;
        wts[i] = p.weights[(int64_t)k * p.C + c0 + cl];
    }
    for (int cl = tid; cl < n_own; cl += FITP_BLOCK) stale[cl] = 1u, pick_of[cl] = draw_pick(cl, p.first_step);
    const int last = p.first_example + p.n_examples - 1;
    int n_now = 0, n_next = 0;          // node counts of example i and i + 1
    uint32_t base_now = 0, base_next = 0;  // node_index of example i and i + 1
    FitGraph fg{};                      // the slot of example i
    if (p.n_examples > 0) {
        n_now = (int)p.n_nodes[p.first_example];
        base_now = p.node_index[p.first_example];
        const int e1 = min(p.first_example + 1, last);
        n_next = (int)p.n_nodes[e1];
        base_next = p.node_index[e1];
        fg = fit_graph_slot(p.tg, p.first_example, n_now);
        if (!DIRECT) {
            FitRowLoader all;
            all.prepare(fg.words, FITP_BLOCK, tid);
            all.request(p.tiles + (int64_t)fg.tile * p.tg.rows * p.tg.tw + fg.word0, p.tg.tw, p.literals + p.n_types + 1, fg.words,
                        rows_both + wave * 64, FITP_BLOCK, tid);
            __builtin_amdgcn_s_waitcnt(FITP_WAIT_VMEM);
        }
        if (DIRECT) {
            for (int at = tid; at < n_now * LA; at += FITP_BLOCK) x_both[at] = p.X[(int64_t)base_now * LA + at];
            if (tid < n_now) types_lds[0][tid] = p.node_type[base_now + tid];
        }
        for (int k = tid; k < K; k += FITP_BLOCK) y_both[k] = (uint32_t)p.encoded_Y[(int64_t)p.first_example * K + k];
    }
    for (int j = tid; j < 6 * K; j += FITP_BLOCK) seen[j] = 0u;
    lds_barrier();

    const int ones_row = p.literals + p.n_types;
    const uint32_t by_words = 0xFFFFFFFFu / (uint32_t)LA, by_bytes = 0xFFFFFFFFu / (uint32_t)(4 * LA);  // (a quotient from them is one too low at most)
    FitRowLoader loader{};
    int loader_words = 0;
    // The threads that add the group's votes to the device-wide class sums and then poll for them are the first K
    // of the LAST wave when K <= 64; that wave requests none of the next graph's words and draws no random
    // numbers, so its polling starts at once and runs beside the other waves' work instead of after its own share.
    const bool poll_apart = K <= 64;
    const int poll0 = poll_apart ? (WAVES - 1) * 64 : 0;         // the first polling thread
    const int loaders = poll_apart ? poll0 : FITP_BLOCK;        // threads 0 .. loaders - 1 request the next graph's words
    const int place = lane & ((1 << p.lanes_log) - 1);
    const bool one_type = p.n_types == 1;
    int slot = 0;  // i modulo 3
    for (int i = 0; i < p.n_examples; ++i) {
        const uint32_t step = p.first_step + (uint32_t)i;
        const uint32_t *rows = rows_both + (i & 1) * p.rows_words;
        const uint32_t *x_now = x_both + (i & 1) * p.x_words;

        // ---- 1. evaluate own clauses (K1 + K7), votes (K6)
        const int stride = fitl_stride(fg.words);
        const uint32_t *col = rows + (2 * place < stride ? 2 * place : 0);  // every group of lanes reads whole rows
        for (int cl = wave; cl < n_own; cl += WAVES) {
            const int c = c0 + cl;
            const uint32_t *inc = ta + (size_t)cl * LA * B + (B - 1);
            uint16_t *list = lists + (size_t)cl * p.lists;
            const uint32_t stale_now = stale[cl];
            const int listed = incl_of[cl];
            const uint32_t state = __builtin_amdgcn_readfirstlane(stale_now);
            int included = __builtin_amdgcn_readfirstlane(listed);
            if (state & 1u) {
                int n = 0;
                if constexpr (!DIRECT) {
                    if (lane == 0 && p.lists > 0) list[0] = (uint16_t)(p.literals + (one_type ? 0 : c % p.n_types));
                    n = 1;
                }
                for (int w0 = 0; w0 < LA; w0 += 64) {
                    uint32_t mine = w0 + lane < LA ? inc[(w0 + lane) * B] : 0u;
                    if (w0 + lane == LA - 1) mine &= p.filter;
                    if constexpr (DIRECT)
                        n += wave_sum_small(__popc(mine));
                    else
                        n = fitl_append(mine, min(64, LA - w0), 32 * w0, list, p.lists, n, lane);
                }
                if constexpr (!DIRECT) fitl_finish(list, p.lists, n, ones_row, p.lanes_log, lane);
                included = DIRECT ? n : n - 1;
                if (lane == 0) incl_of[cl] = included, stale[cl] = 0u;
                fitp_wave_lds_sync();
            } else if (state != 0u && lane == 0) {
                stale[cl] = 0u;
            }
            uint2 v;
            if constexpr (DIRECT) {
                // a few nodes: the clause against each node's own literal words (kernels.py:443-466 as
                // it stands), lane w on word w; no literal-major rows are read or staged
                const uint32_t type = lane < n_now ? types_lds[i & 1][lane] : 0xFFFFFFFFu;
                uint32_t bits = (uint32_t)__ballot((int)type == (one_type ? 0 : c % p.n_types));
                for (int w0 = 0; w0 < LA && bits != 0u; w0 += 64) {
                    const bool there = w0 + lane < LA;
                    uint32_t mine = there ? inc[(w0 + lane) * B] : 0u;
                    if (w0 + lane == LA - 1) mine &= p.filter;
                    const uint32_t *xs = x_now + (there ? w0 + lane : 0);
                    uint32_t violated = 0u;
#pragma unroll 4
                    for (int node = 0; node < n_now; ++node) violated |= (uint32_t)(__ballot((mine & ~xs[node * LA]) != 0u) != 0ull) << node;
                    bits &= ~violated;
                }
                v = make_uint2(lane == 0 ? bits : 0u, 0u);
            } else {
                const uint2 acc = included < p.lists ? fitl_truth(list, included + 1, col, stride, p.lanes_log, lane)
                                                     : fitl_walk(inc, B, LA, p.filter, p.literals + (one_type ? 0 : c % p.n_types),
                                                                 ones_row, col, stride, p.lanes_log, lane);
                v = fitl_nodes(acc, fg, p.lanes_log, lane);
            }
            const int node = n_now == 0 ? -1 : fitl_pick_node(v, pick_of[cl], lane);
            const bool fired = n_now == 0 || node >= 0;  // (the reference's arithmetic for a graph without nodes, kernels.py:289-295)
            if (lane == 0) node_of[cl] = node;
            if (fired)
                for (int k = lane; k < K; k += 64) atomicAdd(&votes[k], wts[cl * K + k]);  // LDS
        }

        // ---- 2. class sums across the device (see the header comment)
        if (tid == 0) go_on = 1;
        lds_barrier();  // the group's votes are complete
        unsigned long long *slot_now = p.class_sum + (size_t)slot * K * FITP_SUM_PARTS * FITP_SUM_STRIDE;
        if (tid >= poll0 && tid - poll0 < K) {  // (K <= FITP_BLOCK: one class per thread)
            const int k = tid - poll0;
            __hip_atomic_fetch_add(&slot_now[(k * FITP_SUM_PARTS + (int)(blockIdx.x % FITP_SUM_PARTS)) * FITP_SUM_STRIDE], FITP_ARRIVED + (unsigned long long)(long long)votes[k], __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
            votes[k] = 0;
        }
        // Work that does not need the class sums is done while the other groups arrive: the next
        // graph's rows, literal words and labels are requested (straight into the other LDS
        // buffers; they are waited for at the end of the step). Nothing is requested before the barrier above: what is
        // under way into LDS has to land before a barrier, and the literal words of the picked nodes, requested as soon as
        // the nodes were known, held that barrier up by their memory latency (6.8 -> 5.9 us per example on 361 nodes).
        const bool has_next = i + 1 < p.n_examples;
        const int ex = p.first_example + i;
        const FitGraph fn = fit_graph_slot(p.tg, has_next ? ex + 1 : ex, has_next ? n_next : n_now);
        // node count and first node of the graph after the next, fetched by two threads and handed over through LDS
        uint32_t after = 0u;
        if (tid < 2) after = (tid == 0 ? p.n_nodes : p.node_index)[min(ex + 2, last)];
        uint32_t type_ahead = 0u;
        if (DIRECT && has_next && tid < n_next) type_ahead = p.node_type[base_next + tid];
        // the literal words of the nodes that the wave's clauses learn from
        if (!DIRECT && p.ahead)
            for (int cl = wave; cl < n_own; cl += WAVES) {
                const int node = __builtin_amdgcn_readfirstlane(node_of[cl]);
                if (node < 0) continue;
                for (int w0 = 0; w0 < LA; w0 += 64)
                    if (w0 + lane < LA) fitp_load_to_lds(p.X + ((int64_t)base_now + node) * LA + w0 + lane, x_ahead + (size_t)cl * LA + w0);
            }
        if constexpr (!DIRECT) {
            if (fn.words != loader_words) loader_words = fn.words, loader.prepare(fn.words, loaders, tid);
            if (has_next)
                loader.request(p.tiles + (int64_t)fn.tile * p.tg.rows * p.tg.tw + fn.word0, p.tg.tw, p.literals + p.n_types + 1, fn.words,
                               rows_both + (~i & 1) * p.rows_words + wave * 64, loaders, tid);
        } else {
            const int next_x_total = has_next ? n_next * LA : 0;
            const uint32_t *src = p.X + (int64_t)base_next * LA + tid;
            uint32_t *dst = x_both + (~i & 1) * p.x_words + wave * 64;
            for (int at0 = 0; at0 < next_x_total && tid < loaders; at0 += loaders)
                if (at0 + tid < next_x_total) fitp_load_to_lds(src + at0, dst + at0);
        }
        if (has_next) {
            const uint32_t *src = (const uint32_t *)p.encoded_Y + (int64_t)(ex + 1) * K + tid;
            uint32_t *dst = y_both + (~i & 1) * K + wave * 64;
            for (int at0 = 0; at0 < K && tid < loaders; at0 += loaders)
                if (at0 + tid < K) fitp_load_to_lds(src + at0, dst + at0);
        }
        // The random words of the feedback gates and of the next step's node picks are drawn by the waves that
        // do not poll, while the class sums are on their way. (Drawing the Type I feedback bits of every (clause, class,
        // word) here as well costs more generator work than the exchange hides: they are drawn
        // afterwards, for the pairs that turn out to need them.)
        const int pollers = (K + 63) & ~63, helpers = FITP_BLOCK - pollers;
        const bool helped = helpers >= FITP_BLOCK / 2;
        // (the polling threads are the first `pollers`, or - set apart - within the last 64)
        if (!helped || (poll_apart ? tid < poll0 : tid >= pollers)) {
            const int first = !helped || poll_apart ? tid : tid - pollers, every = helped ? helpers : FITP_BLOCK;
            for (int j = first; j < n_own * KW; j += every) pos_of[j] = 0u, neg_of[j] = 0u;
            if (first == 0) n_pairs = 0, n_busy = 0;
            for (int j = first; j < n_own * (K + 1); j += every) {
                if (j >= n_own * K) {
                    pick_of[j - n_own * K] = draw_pick(j - n_own * K, step + 1u);
                    continue;
                }
                const int cl = j / K, k = j - cl * K;
                philox_out r = philox4x32_10((uint32_t)(c0 + cl), (uint32_t)k, step, GTM_TAG_CLAUSE_UPDATES, p.k0, p.k1);
                gate[2 * j] = r.v[0];
                gate[2 * j + 1] = r.v[1];
            }
        }
        if (!helped) lds_barrier();
        if (tid >= poll0 && tid - poll0 < K) {
            const int k = tid - poll0;
            const unsigned long long everyone = (unsigned long long)gridDim.x;
            auto arrivals = [](unsigned long long now, unsigned long long before) {
                return ((now - before + FITP_HALF) >> 48) & 0xFFFFull;
            };
            uint32_t *seen_slot = seen + (size_t)slot * 2 * K;
            const unsigned long long seen_own = ((unsigned long long)seen_slot[K + k] << 32) | seen_slot[k];
            uint32_t polls = 0;
            unsigned long long waiting_since = 0ull;
            unsigned long long word = 0ull;
            bool ok = !p.force_abort;
            if (!ok) __hip_atomic_store(p.abort_flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            while (ok) {
                // the abort flag travels with the parts: asked for after a look in vain it was a second round trip per look
                unsigned long long part[FITP_SUM_PARTS];
#pragma unroll
                for (int s = 0; s < FITP_SUM_PARTS; ++s)
                    part[s] = __hip_atomic_load(&slot_now[(k * FITP_SUM_PARTS + s) * FITP_SUM_STRIDE], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                const uint32_t aborted = __hip_atomic_load(p.abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                word = 0ull;
#pragma unroll
                for (int s = 0; s < FITP_SUM_PARTS; ++s) word += part[s];
                if (arrivals(word, seen_own) == everyone) break;
                if (aborted != 0 || fit_wait_is_over(polls, p.spin_limit, waiting_since, p.wait_ticks)) {
                    __hip_atomic_store(p.abort_flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    ok = false;
                    break;
                }
            }
            if (!ok) go_on = 0;
            sums[k] = (int32_t)(long long)(word - seen_own - (everyone << 48));
            // for the slot's next use, three examples on
            seen_slot[k] = (uint32_t)word, seen_slot[K + k] = (uint32_t)(word >> 32);
        }
        __builtin_amdgcn_s_waitcnt(FITP_WAIT_VMEM);  // the next graph's words are in LDS
        if (tid < 2) after_lds[tid] = after;
        if (DIRECT && has_next && tid < n_next) types_lds[(i + 1) & 1][tid] = type_ahead;
        lds_barrier();
        if (!go_on) break;  // uniform over the group; every group leaves at its next check

        // ---- 3. feedback (K8) and automaton updates (K9) on the LDS copies
        const int32_t *y = (const int32_t *)(y_both + (i & 1) * K);
        auto decide = [&](int cl, int k) {  // K8 for a (clause, class) pair
            const int j = cl * K + k;
            int cs = sums[k];
            cs = cs > p.T ? p.T : (cs < -p.T ? -p.T : cs);
            const int yk = y[k];
            const int target = 1 - 2 * (cs > yk);
            int w = wts[j];
            const int sign = (w >= 0) - (w < 0);
            int err = yk - cs;
            err = err < 0 ? -err : err;
            const bool skip = (target == -1 && (uint64_t)gate[2 * j] >= p.q_thr) ||
                              ((uint64_t)gate[2 * j + 1] * (uint64_t)(2 * (int64_t)p.T) >= ((uint64_t)err << 32));
            const int u = skip ? 0 : target * sign;
            const bool fired = node_of[cl] != -1;
            if (u > 0 && fired && (w < 0 ? -(int64_t)w : (int64_t)w) < 2147483647) {
                wts[j] = w + sign;
            } else if (u < 0 && fired) {
                w -= sign;
                if (p.negative == 0 && w < 1) w = 1;
                wts[j] = w;
            }
            return u;
        };
        // word w of the literals of the node that clause cl learns from
        auto literal_word = [&](int cl, int node, int w) {
            if constexpr (DIRECT) return x_now[node * LA + w];
            if (p.ahead) return x_ahead[(size_t)cl * LA + w];
            // (an atomic load, so that the compiler does not make one flat load of the two)
            return __hip_atomic_load(&p.X[((int64_t)base_now + node) * LA + w], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        };
        auto planes_of = [&](int cl, int w) {
            return (uint32_t *)__builtin_assume_aligned(ta + ((size_t)cl * LA + w) * B, EXACT && MAXB == 8 ? 16 : 4);
        };
        for (int j = tid; j < n_own * K; j += FITP_BLOCK) {
            const int cl = j / K, k = j - cl * K;
            const int u = decide(cl, k);
            if (u == 0) continue;
            // listed: the pairs that need Type I bits, and the clauses that get any feedback (once)
            if (u > 0) pair_list[atomicAdd(&n_pairs, 1)] = j;
            atomicOr(&(u > 0 ? pos_of : neg_of)[cl * KW + (k >> 5)], 1u << (k & 31));
            if (atomicOr(&stale[cl], 2u) < 2u) busy_list[atomicAdd(&n_busy, 1)] = cl;
        }
        lds_barrier();
        // a thread per byte of Type I bits (with 2^n threads per pair and clause, half of them idle just above 128 words, an example of
        // 150 words and 1,000 clauses took 11.9 us on single nodes, 9.6 now)
        for (int t = tid; t < n_pairs * 4 * LA; t += FITP_BLOCK) {
            int pair = (int)__umulhi((uint32_t)t, by_bytes), item = t - pair * 4 * LA;
            if (item >= 4 * LA) item -= 4 * LA, ++pair;
            const int j = pair_list[pair], cl = j / K, k = j - cl * K, w = item >> 2, q = item & 3;
            ((uint8_t *)&fbits[((size_t)cl * LA + w) * K + k])[q] =
                (uint8_t)fitl_feedback_byte(p.k0, p.k1, (uint32_t)(c0 + cl), (uint32_t)w, (uint32_t)q, step, 0u, (uint32_t)k, p.thr16);
        }
        lds_barrier();
        for (int t = tid; t < n_busy * LA; t += FITP_BLOCK) {
            int at = (int)__umulhi((uint32_t)t, by_words), w = t - at * LA;
            if (w >= LA) w -= LA, ++at;
            const int cl = busy_list[at];
            const int node = node_of[cl];
            const bool fired = node != -1;
            const bool learns = fired && incl_of[cl] <= p.max_included;
            const uint32_t x = fired ? literal_word(cl, node, w) : 0u;
            fits_word<MAXB, EXACT> word(planes_of(cl, w), B);
            const uint32_t was = word.top();
            const uint32_t *fb_of = fbits + ((size_t)cl * LA + w) * K;
            for (int kw = 0; kw < KW; ++kw)
                fitl_feedback(word, pos_of[cl * KW + kw], neg_of[cl * KW + kw], fired, learns, p.boost, x, fb_of + 32 * kw);
            word.store(planes_of(cl, w));
            if (word.top() != was) atomicOr(&stale[cl], 1u);
        }
        lds_barrier();
        slot = slot == 2 ? 0 : slot + 1;
        fg = fn;
        n_now = n_next;
        base_now = base_next;
        n_next = (int)after_lds[0];
        base_next = after_lds[1];
    }
    __builtin_amdgcn_s_waitcnt(FITP_WAIT_VMEM);  // no load into LDS is left in flight when the group ends
    lds_barrier();
    // own state -> global memory (also after an abort: every clause is left as of some whole step)
    for (int i = tid; i < n_own * LA * B; i += FITP_BLOCK) p.bank[(int64_t)c0 * LA * B + i] = ta[i];
    for (int i = tid; i < n_own * K; i += FITP_BLOCK) {
        int cl = i / K, k = i - cl * K;
        p.weights[(int64_t)k * p.C + c0 + cl] = wts[i];
    }
}
