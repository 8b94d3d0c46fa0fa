// A run of training examples (the loop at tm.py:669-747) of a SMALL model with
// message layers on TINY graphs (at most 64 nodes, MESSAGE_SIZE a multiple of
// 32) as one launch of one workgroup: the automata of every bank, the weights
// and everything a step produces live in LDS, and the phases of a step are
// separated by workgroup barriers only.  At this size a step is a chain of dependent
// instructions, not work: what counts is how many instructions the longest wave of each
// phase runs (a wave issues one in four to five clocks) and which waits are on that chain.
//
// Per example, for the four waves that work (one line per barrier-separated phase):
//   layer 0  K1: a few lanes per (clause, node): (include & ~X[node]) == 0 and the
//            node-type gate (kernels.py:443-466)
//   per message layer
//     send   K3-K5: a thread per (clause, edge), the hypervector bits of a clause true where the
//            edge starts, rotated, straight to its far end; with many edges in two phases,
//            per-node bit vectors (kernels.py:565-588) and the vectors rotated along the edges
//     K2     a few lanes per (clause, node) against the message bank's include
//            words; the negated message literals are the complement of the
//            received vector (kernels.py:505-527)
//   K7, K6, K8  node pick and class sums (kernels.py:319-354, :279-317), feedback decision,
//            weight update (kernels.py:356-405): one wave by itself while it has a lane per
//            (clause, class), else two phases
//   K9, K10  Type I / II on every bank (kernels.py:98-242)
// The random numbers are the same counter-based ones as everywhere else, so the
// result equals the other training paths bit for bit.
//
// A fifth wave helps, in a loop of its own with the same barriers: it fetches the next example (literal
// words, node types, edge counts and offsets, labels; the node count and offset of the one after) and, as soon as
// the offsets are there, its edges - memory latency that nobody waits for -, clears what the phases add to, and
// draws the first 64 random numbers of K7 and K8 while the others pick and decide (where LDS has no room for two
// examples' draws, after that); the four draw the rest after their feedback.  The barriers order LDS traffic only.
//
// Measured on pairs of nodes (10 clauses, 2 + 16 include words each, 2 classes), per example: 5.5 us with one thread
// per pair, run-time divisions and every wave doing all of this; 4.9 with the helper wave, divisions as
// multiplications, the planes of an automaton word known to the compiler and one pass that counts up and down; 3.6
// with the edges requested a step ahead, the draws where the helper idles, and votes and decisions by the same
// threads on values requested together (by clock64, cycles before that: layer 0 3,500 - the edges' latency -, send
// 1,440, K2 1,620, pick to decisions 3,900, feedback 2,600).
#pragma once

constexpr int FITS_BLOCK = 256;                    // threads that work
constexpr int FITS_THREADS = FITS_BLOCK + 64;      // and the helper wave
constexpr int FITS_MAX_NODES = 64;
constexpr size_t FITS_MAX_LDS_BYTES = 128 * 1024;  // of the 160 KB a workgroup can have
// Literal words per helper lane fetched ahead; the rest is read at the step's end, by the four waves that work: graphs of
// 64 nodes of 64 words 14.0 us per example before there was a helper, 17.3 when it read the rest by itself, 9.5 now.
constexpr int FITS_X_AHEAD = 16;
constexpr int FITS_EDGES_LDS = FITS_BLOCK;         // edges of a graph parked in LDS (more: read in place)
// (clause, edge, bit)s per thread up to which messages skip the nodes' vectors.  Chains, us per example, straight | through the
// vectors: 280 in all 5.3 | 6.3, 600 5.7 | 6.1, 1,240 6.7 | 6.7, 2,500 8.0 to 8.2 | 8.0.
constexpr int FITS_DIRECT = 4;
constexpr uint32_t FITS_IS_DIRECT = 1u << 16;      // in what is told of an example's nodes
constexpr int FITS_Y_LDS = 64;                     // classes whose labels are fetched ahead (K <= this, else read in place)

struct FitSmallParams {
    // data set
    const uint32_t *X, *node_type, *node_index, *n_nodes, *n_edges, *edge_index, *edge;
    const int32_t *encoded_Y;
    int first_example, n_examples;
    uint32_t first_step;
    int n_types, has_edges;
    // model
    uint32_t *bank[GTM_MAX_DEPTH];     // bank 0: literals of the nodes; bank l: message literals of layer l
    uint32_t filter[GTM_MAX_DEPTH];    // valid bits of a bank's last include word
    uint32_t thr16[GTM_MAX_DEPTH];
    int32_t *weights;                  // [K][C]
    const uint32_t *hv;                // [C][MB]
    int depth, C, LA, MC, MW, MB, B, K, T, negative, boost, max_included;
    uint32_t k0, k1;
    uint64_t q_thr;
    // how the work is spread (fit_small_lanes)
    int lanes0, lanes1;         // log2 of the lanes that share a (clause, node): layer 0, message layers
    int inc_copy;               // the include planes have a copy of their own in LDS
    int draws_twice;            // the random draws of two examples have room in LDS: the next one's need not wait
    uint32_t by_LA, by_MC, by_MW, by_K, by_types;  // fits_magic of these
};

// j / d as a multiplication: exact where j d < 2^32, which LDS sizes see to.  A run-time division is 25 dependent
// instructions, and a step had a dozen of them on its one chain.
__host__ __device__ __forceinline__ uint32_t fits_magic(uint32_t d) { return d > 1 ? 0xFFFFFFFFu / d + 1u : 0u; }
__device__ __forceinline__ int fits_div(int j, int d, uint32_t magic) { return d == 1 ? j : (int)__umulhi((uint32_t)j, magic); }

// LDS words the kernel needs (the host checks it against the limit it sets).
inline size_t fit_small_lds_words(int depth, int C, int LA, int MC, int MW, int MB, int B, int K) {
    const size_t banks = (size_t)C * (LA + (size_t)(depth - 1) * MC) * B;
    return banks + (size_t)K * C                              // weights
           + (size_t)C * MB                                   // hypervector bits
           + 2 * ((size_t)FITS_MAX_NODES * LA + 3 * FITS_MAX_NODES + FITS_Y_LDS + 2)  // graph data, two examples
           + 2 * (size_t)FITS_EDGES_LDS                       // edges
           + 2 * (size_t)C * 2                                // truth of two layers, 2 words per clause
           + (size_t)depth * FITS_MAX_NODES * MW              // sent; got per layer
           + (size_t)K + 2 * (size_t)C + (size_t)C * K        // class sums, picked node, include count, updates
           + (size_t)C + 2 * (size_t)C * K;                   // random draws of K7 and K8
}

// ... and what came to that: the second half of the include counts, the table of fits_magic and what is known of an
// example (twice); where there is room, the second half of the random draws and the include planes' copy (else the
// planes are read where they are).
inline size_t fit_small_lds_more_words(int depth, int C, int LA, int MC, int K, bool draws_twice, bool inc_copy) {
    return (size_t)C + FITS_EDGES_LDS + 1 + 8 + (draws_twice ? (size_t)C + 2 * (size_t)C * K : 0) +
           (inc_copy ? (size_t)C * (LA + (size_t)(depth - 1) * MC) : 0);
}

// log2 of the lanes that share a (clause, node) of `words` include words: as many as the workgroup has for the pairs
// of the largest graph, at most 16 and at most the words.
inline int fit_small_lanes(int C, int max_nodes, int words) {
    int lg = 0;
    while (lg < 4 && (2 << lg) <= words && ((int64_t)C * max_nodes << (lg + 1)) <= FITS_BLOCK) ++lg;
    return lg;
}

// This lane's words (part, part + lanes, ...) of a clause's include words against a node's literal words: the violated
// bits ORed together; adds the number of included literals.  MESSAGES: include word w >= half is held against
// the complement of literal word w - half (message banks).  Four words are in flight at a time.
// HALVES: both halves divide into such groups of four, so that no word is asked which half it is in, or whether it is there
// (nor for its valid bits: message sizes are multiples of 32 here).
// It is a form of the kernel of its own: chosen in here, by sizes, it cost pairs of nodes 0.15 us per example.
template <bool MESSAGES, bool HALVES>
__device__ __forceinline__ uint32_t fits_violations(const uint32_t *inc, int stride, const uint32_t *x, int n_words, int half,
                                                     uint32_t last_filter, int part, int lanes, int *included) {
    uint32_t bad = 0u;
    int count = 0;
    if constexpr (HALVES) {
        for (int side = 0; side < 2; ++side, inc += half * stride) {
            const uint32_t flip = side == 0 ? 0xFFFFFFFFu : 0u;
            for (int w0 = part; w0 < half; w0 += 4 * lanes) {
                uint32_t i[4], v[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) i[u] = inc[(w0 + u * lanes) * stride], v[u] = x[w0 + u * lanes] ^ flip;
#pragma unroll
                for (int u = 0; u < 4; ++u) bad |= i[u] & v[u], count += __popc(i[u]);
            }
        }
        *included += count;
        return bad;
    }
    for (int w0 = part; w0 < n_words; w0 += 4 * lanes) {
        uint32_t i[4], v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int w = w0 + u * lanes, at = w < n_words ? w : part;
            const bool negated = MESSAGES && at >= half;
            i[u] = inc[at * stride];
            v[u] = x[negated ? at - half : at];
            if (negated) v[u] = ~v[u];
            if (w >= n_words) i[u] = 0u;
            if (w == n_words - 1) i[u] &= last_filter;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) bad |= i[u] & ~v[u], count += __popc(i[u]);
    }
    *included += count;
    return bad;
}

// Is `has` false in all 2^k neighbouring lanes (an aligned group) that share a (clause, node)?
__device__ __forceinline__ bool fits_group_has_none(bool has, int lane, int lanes) {
    const unsigned long long all = __ballot(has);
    return ((all >> (lane & ~(lanes - 1))) & ((1ull << lanes) - 1ull)) == 0ull;
}

// The planes of one automaton word in registers.  EXACT: MAXB of them, known to the compiler (the default, 8), else B.
template <int MAXB, bool EXACT>
struct fits_word {
    uint32_t ta[MAXB];
    const int B;
    __device__ __forceinline__ fits_word(const uint32_t *from, int planes) : B(planes) {
#pragma unroll
        for (int b = 0; b < MAXB; ++b) ta[b] = EXACT || b < B ? from[b] : 0u;
    }
    __device__ __forceinline__ uint32_t top() const {
        uint32_t t = ta[MAXB - 1];
        if (!EXACT) {
#pragma unroll
            for (int b = 0; b < MAXB; ++b)
                if (b == B - 1) t = ta[b];
        }
        return t;
    }
    // Automata of `up` one state up, those of `down` (no common bits) one down, both stopping at the ends: one pass
    // over the planes, whichever of the two a lane needs.
    __device__ __forceinline__ void count(uint32_t up, uint32_t down) {
#pragma unroll
        for (int b = 0; b < MAXB; ++b)
            if (EXACT || b < B) {
                const uint32_t v = ta[b];
                ta[b] = v ^ (up | down);
                up &= v, down &= ~v;
            }
#pragma unroll
        for (int b = 0; b < MAXB; ++b)
            if (EXACT || b < B) ta[b] = (ta[b] | up) & ~down;
    }
    __device__ __forceinline__ void store(uint32_t *to) const {
#pragma unroll
        for (int b = 0; b < MAXB; ++b)
            if (EXACT || b < B) to[b] = ta[b];
    }
};

// Four waves work, the fifth (`helper`) fetches: each has a loop of its own over the examples, with the same barriers.
template <int MAXB, bool EXACT, bool HALVES>
__global__ __launch_bounds__(FITS_THREADS) void k_fit_small(FitSmallParams p) {
    // An array of its own name, so that the other kernels' `lds`, which is known to lie on 16 bytes, is not taken for it: an automaton word's planes
    // in two 128-bit accesses, 32 bytes from lane to lane, make an example longer than in four pairs of words (49 clauses 6.83 us, 6.59 in pairs).
    extern __shared__ uint32_t fits_lds[];
    const int tid = threadIdx.x;
    const int C = p.C, LA = p.LA, MC = p.MC, MW = p.MW, B = EXACT ? MAXB : p.B, K = p.K, layers = p.depth - 1;

    // LDS carve-up: bank 0, then the message banks (all of one size), then the rest
    const size_t bank0_words = (size_t)C * LA * B, message_bank_words = (size_t)C * MC * B;
    auto bank_of = [&](int l) { return l == 0 ? fits_lds : fits_lds + bank0_words + (size_t)(l - 1) * message_bank_words; };
    int32_t *wts = (int32_t *)(fits_lds + bank0_words + (size_t)layers * message_bank_words);  // [K][C]
    uint32_t *hv = (uint32_t *)(wts + K * C);      // [C][MB]
    // per example, double-buffered: literal words [nodes][LA]; node type, edge count, first edge
    // [3][nodes]; labels [FITS_Y_LDS]; node count and first node of the example after
    const int graph_words = FITS_MAX_NODES * LA + 3 * FITS_MAX_NODES + FITS_Y_LDS + 2;
    uint32_t *graph_buf = hv + C * p.MB;
    uint32_t *edges_lds = graph_buf + 2 * graph_words;  // [FITS_EDGES_LDS][2]
    uint32_t *truth[2] = {edges_lds + 2 * FITS_EDGES_LDS, edges_lds + 2 * FITS_EDGES_LDS + 2 * C};  // [C][2]
    uint32_t *sent = truth[1] + 2 * C;             // [nodes][MW]
    uint32_t *got_all = sent + FITS_MAX_NODES * MW;  // [layers][nodes][MW]: what each node received, per layer
    int32_t *sums = (int32_t *)(got_all + (size_t)layers * FITS_MAX_NODES * MW);  // [K]
    int32_t *node_of = sums + K;                   // [C]
    int32_t *incl_both = node_of + C;              // [2][C], the second half for odd examples
    int32_t *upd = incl_both + 2 * C;              // [C][K]
    const int draw_words = p.draws_twice ? C + 2 * C * K : 0;  // (from an example's to the next one's)
    uint32_t *draw_both = (uint32_t *)(upd + C * K);  // [C] node picks, [C][K][2] decisions
    // twice: an example's nodes and FITS_IS_DIRECT, edges, first edge (of direct ones the edges' magic), magic of its nodes
    uint32_t *info_both = draw_both + C + 2 * C * K + draw_words;
    uint32_t *magic_of = info_both + 8;            // [FITS_EDGES_LDS + 1]
    // the include planes, every bank's words in order: a copy, so that lanes read neighbouring words, or in place
    uint32_t *inc_copy = magic_of + FITS_EDGES_LDS + 1;
    const uint32_t *inc_words = p.inc_copy ? inc_copy : fits_lds + (B - 1);
    const int inc_stride = p.inc_copy ? 1 : B;
    const int all_words = C * (LA + layers * MC);
    const int lane = tid & 63;
    const bool one_wave = C <= 64 && C * K <= 64;  // node pick, votes and decisions by wave 0 alone, no barrier between them

    const int draws = C + C * K;
    // one generator call per draw of example i: draws first, first + stride, ...
    auto draw = [&](int i, int first, int end, int stride) {
        const uint32_t at_step = p.first_step + (uint32_t)i;
        uint32_t *draw_node = draw_both + (i & 1) * draw_words, *draw_update = draw_node + C;
        for (int j = first; j < end; j += stride) {
            const bool pick = j < C;
            const int ck = pick ? 0 : j - C, c = pick ? j : fits_div(ck, K, p.by_K), k = pick ? 0 : ck - c * K;
            const philox_out r = philox4x32_10<false>((uint32_t)c, (uint32_t)k, at_step, pick ? GTM_TAG_CLAUSE_NODE : GTM_TAG_CLAUSE_UPDATES, p.k0, p.k1);
            uint32_t *to = pick ? draw_node + j : draw_update + 2 * ck;
            to[0] = r.v[0];
            if (!pick) to[1] = r.v[1];
        }
    };
    struct Example {  // where example i's data are
        uint32_t *x_rows, *types, *ne, *ei, *labels, *header;
    };
    auto example = [&](int i) {
        Example e;
        e.x_rows = graph_buf + (i & 1) * graph_words;
        e.types = e.x_rows + FITS_MAX_NODES * LA;
        e.ne = e.types + FITS_MAX_NODES, e.ei = e.types + 2 * FITS_MAX_NODES;
        e.labels = e.types + 3 * FITS_MAX_NODES, e.header = e.labels + FITS_Y_LDS;
        return e;
    };
    auto tell = [&](int i, int nodes, int edges, bool direct, uint32_t first_edge) {  // (one lane)
        uint32_t *info = info_both + 4 * (i & 1);
        info[0] = (uint32_t)nodes | (direct ? FITS_IS_DIRECT : 0u);
        info[1] = (uint32_t)edges, info[2] = direct ? magic_of[edges > 0 ? edges : 1] : first_edge;
        info[3] = magic_of[nodes > 0 ? nodes : 1];
    };

    // state -> LDS
    for (int l = 0; l < p.depth; ++l) {
        uint32_t *dst = bank_of(l);
        const uint32_t *src = p.bank[l];
        for (int i = tid; i < C * (l == 0 ? LA : MC) * B; i += FITS_THREADS) dst[i] = src[i];
    }
    if (p.inc_copy)
        for (int l = 0; l < p.depth; ++l) {
            const int first = l == 0 ? 0 : C * LA + (l - 1) * C * MC;
            for (int i = tid; i < C * (l == 0 ? LA : MC); i += FITS_THREADS) inc_copy[first + i] = p.bank[l][(int64_t)i * B + B - 1];
        }
    for (int i = tid; i <= FITS_EDGES_LDS; i += FITS_THREADS) magic_of[i] = fits_magic((uint32_t)i);
    for (int i = tid; i < 2 * C; i += FITS_THREADS) incl_both[i] = 0;
    draw(0, tid, draws, FITS_THREADS);
    for (int i = tid; i < K * C; i += FITS_THREADS) wts[i] = p.weights[i];
    for (int i = tid; i < C * p.MB; i += FITS_THREADS) hv[i] = p.hv[i];
    for (int i = tid; i < 4 * C; i += FITS_THREADS) truth[0][i] = 0u;
    for (int k = tid; k < K; k += FITS_THREADS) sums[k] = 0;
    for (int i = tid; i < FITS_MAX_NODES * MW; i += FITS_THREADS) sent[i] = 0u;

    // the first example's data, and the second's node count and offset
    int n_nodes = (int)p.n_nodes[p.first_example];
    {
        const int64_t base = p.node_index[p.first_example];
        const Example e = example(0);
        for (int j = tid; j < n_nodes * LA; j += FITS_THREADS) e.x_rows[j] = p.X[base * LA + j];
        for (int j = tid; j < n_nodes; j += FITS_THREADS) {
            e.types[j] = p.node_type[base + j];
            e.ne[j] = p.has_edges ? p.n_edges[base + j] : 0u;
            e.ei[j] = p.has_edges ? p.edge_index[base + j] : 0u;
        }
        for (int k = tid; k < K && k < FITS_Y_LDS; k += FITS_THREADS)
            e.labels[k] = (uint32_t)p.encoded_Y[(int64_t)p.first_example * K + k];
        if (tid < 2 && p.n_examples > 1)
            e.header[tid] = (tid == 0 ? p.n_nodes : p.node_index)[p.first_example + 1];
    }
    lds_barrier();

    if (tid >= FITS_BLOCK) {
        // ================ the helper wave
        // The edges of an example travel for most of the example before it (they were 1 us of every step when they were
        // requested at its top): the edge counts and offsets that say where they are came with the example's other data.
        uint32_t first_edge = 0u;
        int graph_edges = 0;
        bool direct = true;
        uint2 edge_ahead[FITS_EDGES_LDS / 64];
        auto request_edges = [&](int nodes, uint32_t count, uint32_t offset) {  // count, offset: of node `lane`
            first_edge = 0u, graph_edges = 0, direct = true;
            if (!p.has_edges || nodes == 0) return;
            first_edge = (uint32_t)__builtin_amdgcn_readfirstlane((int)offset);
            graph_edges = __builtin_amdgcn_readlane((int)(offset + count), nodes - 1) - (int)first_edge;
            // edges that do not lie node after node are not parked but read where they are
            const uint32_t next_offset = (uint32_t)__shfl_down((int)offset, 1);
            if (__ballot(lane < nodes - 1 && next_offset != offset + count) != 0ull) graph_edges = FITS_EDGES_LDS + 1;
            // Few edges: a true clause's bits go straight to the far ends of the edges, a thread per (clause, edge); else
            // through the vectors that the nodes send, one phase more.
            direct = graph_edges <= FITS_EDGES_LDS && (int64_t)graph_edges * C * p.MB <= FITS_DIRECT * FITS_BLOCK;
            const uint2 *from = (const uint2 *)p.edge + first_edge;
            if (graph_edges <= FITS_EDGES_LDS) {
#pragma unroll
                for (int r = 0; r < FITS_EDGES_LDS / 64; ++r)
                    if (64 * r < graph_edges && lane + 64 * r < graph_edges) edge_ahead[r] = from[lane + 64 * r];
            }
        };
        {
            const Example e = example(0);
            request_edges(n_nodes, lane < n_nodes ? e.ne[lane] : 0u, lane < n_nodes ? e.ei[lane] : 0u);
            if (lane == 0) tell(0, n_nodes, graph_edges, direct, first_edge);
        }
        lds_barrier();
        for (int i = 0; i < p.n_examples; ++i) {
            const int ex = p.first_example + i;
            const int nn = n_nodes > 0 ? n_nodes : 1;
            const Example e = example(i), to = example(i + 1);
            const bool direct_now = direct;  // (this example's: the next one's edges are asked for below)
            for (int l = 0; l < layers; ++l)  // (what arrives is ORed in)
                for (int j = lane; j < nn * MW; j += 64) got_all[l * FITS_MAX_NODES * MW + j] = 0u;
            if (graph_edges <= FITS_EDGES_LDS) {
#pragma unroll
                for (int r = 0; r < FITS_EDGES_LDS / 64; ++r) {
                    const int j = lane + 64 * r;
                    if (64 * r < graph_edges && j < graph_edges) {
                        // where messages go straight along the edges, the node that each starts from - the last one whose
                        // first edge is not behind it - in the upper half of the word with the far end
                        uint32_t source = 0u;
                        if (direct_now)
                            for (int ahead = n_nodes > 1 ? 1 << (31 - __clz(n_nodes - 1)) : 0; ahead > 0; ahead >>= 1) {
                                const uint32_t n = source + (uint32_t)ahead;
                                if (n < (uint32_t)n_nodes && e.ei[n] - first_edge <= (uint32_t)j) source = n;
                            }
                        edges_lds[2 * j] = edge_ahead[r].x | (source << 16), edges_lds[2 * j + 1] = edge_ahead[r].y;
                    }
                }
            }
            // what lands at the step's end: example i + 1 (its node count and offset came with example i), the header of i + 2
            const bool more = i + 1 < p.n_examples;
            const int n_next = more ? __builtin_amdgcn_readfirstlane((int)e.header[0]) : 0;
            const int64_t base_next = more ? (int64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)e.header[1]) : 0;
            const int x_words = n_next * LA;
            const uint32_t *x_from = p.X + base_next * LA;
            uint32_t x_ahead[FITS_X_AHEAD], field_ahead[3] = {0u, 0u, 0u}, label_ahead = 0u, header_ahead = 0u;
#pragma unroll
            for (int r = 0; r < FITS_X_AHEAD; ++r)
                if (64 * r < x_words) x_ahead[r] = lane + 64 * r < x_words ? x_from[lane + 64 * r] : 0u;
            if (lane < n_next) {
                field_ahead[0] = p.node_type[base_next + lane];
                if (p.has_edges) field_ahead[1] = p.n_edges[base_next + lane], field_ahead[2] = p.edge_index[base_next + lane];
            }
            if (more && lane < K) label_ahead = (uint32_t)p.encoded_Y[(int64_t)(ex + 1) * K + lane];
            if (lane < 2 && i + 2 < p.n_examples) header_ahead = (lane == 0 ? p.n_nodes : p.node_index)[ex + 2];
            lds_barrier();  // layer 0
            for (int l = 0; l < layers; ++l) {
                // (the rows of truth that the evaluation before this layer's read: free since its barrier)
                if (l > 0)
                    for (int j = lane; j < 2 * C; j += 64) truth[(l & 1) ^ 1][j] = 0u;
                lds_barrier();  // sent
                if (!direct_now) lds_barrier();  // along the edges
                if (!direct_now)
                    for (int j = lane; j < nn * MW; j += 64) sent[j] = 0u;
                lds_barrier();  // K2
            }
            // the longest phase of the others, and the helper's for what takes time
            if (more) {
                if (p.draws_twice) draw(i + 1, lane, min(draws, 64), 64);
                request_edges(n_next, field_ahead[1], field_ahead[2]);
            } else {
                graph_edges = 0;
            }
            for (int j = lane; j < C; j += 64) incl_both[((i + 1) & 1) * C + j] = 0;
            if (!one_wave) lds_barrier();  // votes
            lds_barrier();                 // decisions
            if (more && !p.draws_twice) draw(i + 1, lane, min(draws, 64), 64);
            for (int k = lane; k < K; k += 64) sums[k] = 0;
            for (int j = lane; j < 4 * C; j += 64) truth[0][j] = 0u;  // (both layers' truth: one after the other)
            // example i + 1 lands in the other buffer
#pragma unroll
            for (int r = 0; r < FITS_X_AHEAD; ++r)
                if (64 * r < x_words && lane + 64 * r < x_words) to.x_rows[lane + 64 * r] = x_ahead[r];
            to.types[lane] = field_ahead[0], to.ne[lane] = field_ahead[1], to.ei[lane] = field_ahead[2];
            to.labels[lane] = label_ahead;
            if (lane < 2) to.header[lane] = header_ahead;
            if (lane == 0) tell(i + 1, n_next, graph_edges, direct, first_edge);
            n_nodes = n_next;
            lds_barrier();
        }
    } else {
    // ================ the four that work
    lds_barrier();
    for (int i = 0; i < p.n_examples; ++i) {
        const int ex = p.first_example + i;
        const uint32_t step = p.first_step + (uint32_t)i;
        const uint32_t *info = info_both + 4 * (i & 1);
        const int graph_edges = __builtin_amdgcn_readfirstlane((int)info[1]);
        const uint32_t first_edge = info[2], by_edges = info[2], by_nn = info[3];
        n_nodes = __builtin_amdgcn_readfirstlane((int)info[0]);
        const bool direct = ((uint32_t)n_nodes & FITS_IS_DIRECT) != 0u;
        n_nodes &= (int)(FITS_IS_DIRECT - 1u);
        const int nn = n_nodes > 0 ? n_nodes : 1;  // a graph without nodes: one stand-in pair per clause
        const Example e_now = example(i);
        const uint32_t *x_rows = e_now.x_rows, *types = e_now.types, *ne_lds = e_now.ne, *ei_lds = e_now.ei;
        const int32_t *y = (const int32_t *)e_now.labels;
        const int x_words_next = __builtin_amdgcn_readfirstlane((int)e_now.header[0]) * LA;  // (of no use in the last example)
        const uint32_t *draw_node = draw_both + (i & 1) * draw_words, *draw_update = draw_node + C;
        int32_t *incl_of = incl_both + (i & 1) * C;
        const bool edges_parked = graph_edges <= FITS_EDGES_LDS;

        // ---- layer 0 (K1), 2^lanes0 lanes per (clause, node); truth[0] is all zero here
        uint32_t *cur = truth[0], *nxt = truth[1];
        {
            const int lanes = 1 << p.lanes0, part = tid & (lanes - 1);
            for (int j = tid >> p.lanes0; j < C * nn; j += FITS_BLOCK >> p.lanes0) {
                const int c = fits_div(j, nn, by_nn), n = j - c * nn;
                const int type = p.n_types == 1 ? 0 : c - fits_div(c, p.n_types, p.by_types) * p.n_types;
                const bool match = n_nodes > 0 && (int)types[n] == type;
                if (match || n == 0) {
                    int included = 0;
                    const uint32_t bad = fits_violations<false, false>(inc_words + c * LA * inc_stride, inc_stride, x_rows + n * LA, LA, LA,
                                                                p.filter[0], part, lanes, &included);
                    if (n == 0 && included) atomicAdd(&incl_of[c], included);
                    const bool holds = fits_group_has_none(bad != 0u, lane, lanes);
                    // a graph without nodes: the reference's arithmetic leaves every clause true (kernels.py:289-295)
                    if (part == 0) {
                        if (n_nodes == 0)
                            cur[2 * c] = 0xFFFFFFFFu;
                        else if (match && holds)
                            atomicOr(&cur[2 * c + (n >> 5)], 1u << (n & 31));
                    }
                }
            }
        }
        lds_barrier();

        // ---- message layers; sent is all zero at the start of each
        for (int l = 0; l < layers; ++l) {
            uint32_t *got = got_all + (size_t)l * FITS_MAX_NODES * MW;
            if (direct) {
                for (int j = tid; j < C * graph_edges; j += FITS_BLOCK) {
                    const int c = fits_div(j, graph_edges, by_edges), e = j - c * graph_edges;
                    const uint32_t ends = edges_lds[2 * e], n = ends >> 16, dst = ends & 0xFFFFu;
                    uint32_t type = edges_lds[2 * e + 1];
                    if (!((cur[2 * c + (n >> 5)] >> (n & 31)) & 1u)) continue;
                    if (type >= (uint32_t)(MW * 32)) type %= (uint32_t)(MW * 32);
                    for (int b = 0; b < p.MB; ++b) {
                        uint32_t h = hv[c * p.MB + b] + type;
                        h -= h >= (uint32_t)(MW * 32) ? (uint32_t)(MW * 32) : 0u;
                        atomicOr(&got[dst * MW + (h >> 5)], 1u << (h & 31));
                    }
                }
                lds_barrier();
            } else {
                // what each node sends: the hypervector bits of the clauses true at it
                for (int j = tid; j < C * n_nodes; j += FITS_BLOCK) {
                    const int c = fits_div(j, nn, by_nn), n = j - c * nn;
                    if ((cur[2 * c + (n >> 5)] >> (n & 31)) & 1u)
                        for (int b = 0; b < p.MB; ++b) {
                            const uint32_t h = hv[c * p.MB + b];
                            atomicOr(&sent[n * MW + (h >> 5)], 1u << (h & 31));
                        }
                }
                lds_barrier();
                // along every edge: the vector rotated by the edge type (bit p of the result is bit (p - type) mod M)
                if (graph_edges > 0)
                    for (int j = tid; j < n_nodes * MW; j += FITS_BLOCK) {
                        const int n = fits_div(j, MW, p.by_MW), jw = j - n * MW;
                        const uint32_t ne = ne_lds[n];
                        const uint32_t *v = sent + n * MW;
                        for (uint32_t e = 0; e < ne; ++e) {
                            uint32_t dst, type;
                            if (edges_parked) {
                                const uint32_t at = ei_lds[n] - (uint32_t)first_edge + e;
                                dst = edges_lds[2 * at];
                                type = edges_lds[2 * at + 1];
                            } else {
                                dst = p.edge[((int64_t)ei_lds[n] + e) * 2];
                                type = p.edge[((int64_t)ei_lds[n] + e) * 2 + 1];
                            }
                            const uint32_t shift = type < (uint32_t)(MW * 32) ? type : type % (uint32_t)(MW * 32);
                            const int q = (int)(shift >> 5), r = (int)(shift & 31u);
                            const int a = jw - q + (jw < q ? MW : 0), below = (a > 0 ? a : MW) - 1;
                            const uint32_t word = r ? (v[a] << r) | (v[below] >> (32 - r)) : v[a];
                            if (word) atomicOr(&got[dst * MW + jw], word);
                        }
                    }
                lds_barrier();
            }
            // K2, 2^lanes1 lanes per (clause, node): include words 0 .. MW - 1 against the received
            // vector, MW .. 2 MW - 1 against its complement
            {
                const int lanes = 1 << p.lanes1, part = tid & (lanes - 1);
                const uint32_t *inc_l = inc_words + (C * LA + l * C * MC) * inc_stride;
                for (int j = tid >> p.lanes1; j < C * nn; j += FITS_BLOCK >> p.lanes1) {
                    const int c = fits_div(j, nn, by_nn), n = j - c * nn;
                    const bool alive = n_nodes > 0 && ((cur[2 * c + (n >> 5)] >> (n & 31)) & 1u);
                    if (alive || n == 0) {
                        int included = 0;
                        const uint32_t bad = fits_violations<true, HALVES>(inc_l + c * MC * inc_stride, inc_stride, got + n * MW, MC, MW,
                                                                   p.filter[l + 1], part, lanes, &included);
                        if (n == 0 && included) atomicAdd(&incl_of[c], included);
                        const bool holds = fits_group_has_none(bad != 0u, lane, lanes);
                        if (part == 0) {
                            if (n_nodes == 0)
                                nxt[2 * c] = 0xFFFFFFFFu;
                            else if (alive && holds)
                                atomicOr(&nxt[2 * c + (n >> 5)], 1u << (n & 31));
                        }
                    }
                }
            }
            lds_barrier();
            uint32_t *swap = cur;
            cur = nxt;
            nxt = swap;
        }

        // ---- K7, K6, K8: node pick, class sums; then feedback decisions and weights, one thread per (clause, class).
        // Everything a thread reads is requested at once, and what it read for its vote serves its decision.
        auto true_nodes = [&](int c, unsigned long long *bits) {
            *bits = ((unsigned long long)cur[2 * c + 1] << 32) | cur[2 * c];
            return __popcll(*bits);
        };
        auto pick_node = [&](unsigned long long bits, int count, uint32_t random) {
            if (n_nodes == 0 || count == 0) return -1;
            const int pick = (int)(((uint64_t)random * (uint64_t)count) >> 32);
            for (int j = 0; j < pick; ++j) bits &= bits - 1;
            return __ffsll((long long)bits) - 1;
        };
        auto decide = [&](int j, int c, int k, int w, int yk, uint32_t r0, uint32_t r1, int cs, bool picked) {
            cs = cs > p.T ? p.T : (cs < -p.T ? -p.T : cs);
            const int target = 1 - 2 * (cs > yk);
            const int sign = (w >= 0) - (w < 0);
            int err = yk - cs;
            err = err < 0 ? -err : err;
            const bool skip = (target == -1 && (uint64_t)r0 >= p.q_thr) ||
                              ((uint64_t)r1 * (uint64_t)(2 * (int64_t)p.T) >= ((uint64_t)err << 32));
            const int u = skip ? 0 : target * sign;
            if (u > 0 && picked && (w < 0 ? -(int64_t)w : (int64_t)w) < 2147483647) {
                wts[k * C + c] = w + sign;
            } else if (u < 0 && picked) {
                w -= sign;
                if (p.negative == 0 && w < 1) w = 1;
                wts[k * C + c] = w;
            }
            upd[j] = u;
        };
        const int32_t *y_now = K <= FITS_Y_LDS ? y : p.encoded_Y + (int64_t)ex * K;
        if (one_wave) {
            if (tid < C * K) {
                const int c = fits_div(tid, K, p.by_K), k = tid - c * K;
                const int w = wts[k * C + c], yk = y_now[k];
                const uint32_t random = draw_node[c], r0 = draw_update[2 * tid], r1 = draw_update[2 * tid + 1];
                unsigned long long bits;
                const int count = true_nodes(c, &bits);
                if (n_nodes == 0 || count > 0) atomicAdd(&sums[k], w);
                const bool picked = n_nodes > 0 && count > 0;
                if (k == 0) node_of[c] = pick_node(bits, count, random);
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup", "local");  // (one wave's LDS operations are carried out in order)
                decide(tid, c, k, w, yk, r0, r1, sums[k], picked);
            }
        } else {
            for (int c = tid; c < C; c += FITS_BLOCK) {
                unsigned long long bits;
                const int count = true_nodes(c, &bits);
                node_of[c] = pick_node(bits, count, draw_node[c]);
                if (n_nodes == 0 || count > 0)
                    for (int k = 0; k < K; ++k) atomicAdd(&sums[k], wts[k * C + c]);
            }
            lds_barrier();
            for (int j = tid; j < C * K; j += FITS_BLOCK) {
                const int c = fits_div(j, K, p.by_K), k = j - c * K;
                decide(j, c, k, wts[k * C + c], y_now[k], draw_update[2 * j], draw_update[2 * j + 1], sums[k], node_of[c] != -1);
            }
        }
        lds_barrier();

        // ---- K9, K10: one thread per (clause, automaton word of any bank)
        for (int j = tid; j < all_words; j += FITS_BLOCK) {
            int l = 0, at = j;
            if (at >= C * LA) {
                at -= C * LA, l = 1;
                while (at >= C * MC) at -= C * MC, ++l;
            }
            const int chunks = l == 0 ? LA : MC;
            const int c = fits_div(at, chunks, l == 0 ? p.by_LA : p.by_MC), w = at - c * chunks;
            const int32_t *u_of = upd + c * K;
            int u = u_of[0];
            bool any = u != 0;
            for (int k = 1; k < K; ++k) any |= u_of[k] != 0;
            if (!any) continue;
            const int node = node_of[c];
            const bool fired = node != -1, within = incl_of[c] <= p.max_included, learns = fired && within;
            uint32_t x = 0u;
            if (fired) {
                const uint32_t *got = got_all + (l - 1) * FITS_MAX_NODES * MW + node * MW;
                x = l == 0 ? x_rows[node * LA + w] : w < MW ? got[w] : ~got[w - MW];
            }
            uint32_t thr16 = p.thr16[0];
#pragma unroll
            for (int t = 1; t < GTM_MAX_DEPTH; ++t)
                if (t == l) thr16 = p.thr16[t];
            fits_word<MAXB, EXACT> word(fits_lds + j * B, B);
            for (int k = 0; k < K; ++k) {
                const int now = u;
                if (k + 1 < K) u = u_of[k + 1];
                if (now == 0) continue;
                // Type I where u > 0 (kernels.py:141-173), Type II where u < 0 (:174-183): bits to count up and down
                uint32_t up = fired ? ~x & ~word.top() : 0u, down = 0u;
                if (now > 0) {
                    const uint32_t fb = gtm_feedback_bits<false>(p.k0, p.k1, (uint32_t)c, (uint32_t)w, step, (uint32_t)l, (uint32_t)k, thr16);
                    up = learns ? (p.boost == 1 ? x : x & ~fb) : 0u;
                    down = learns ? ~x & fb : fb;
                }
                word.count(up, down);
            }
            word.store(fits_lds + j * B);
            if (p.inc_copy) inc_copy[j] = word.top();
        }
        // the next example's random numbers: the first 64 are the helper's
        if (i + 1 < p.n_examples) {
            draw(i + 1, 64 + FITS_BLOCK - 1 - tid, draws, FITS_BLOCK);
            // ... and the literal words that the helper does not fetch ahead
            if (x_words_next > 64 * FITS_X_AHEAD) {
                const uint32_t *x_from = p.X + (int64_t)e_now.header[1] * LA;
                uint32_t *to = example(i + 1).x_rows;
                for (int j = tid + 64 * FITS_X_AHEAD; j < x_words_next; j += FITS_BLOCK) to[j] = x_from[j];
            }
        }
        lds_barrier();
    }
    }

    // state -> global memory
    for (int l = 0; l < p.depth; ++l) {
        const uint32_t *src = bank_of(l);
        uint32_t *dst = p.bank[l];
        for (int i = tid; i < C * (l == 0 ? LA : MC) * B; i += FITS_THREADS) dst[i] = src[i];
    }
    for (int i = tid; i < K * C; i += FITS_THREADS) p.weights[i] = wts[i];
}
