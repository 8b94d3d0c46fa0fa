// Class sums of small models on tiny graphs in one launch (`_score`, tm.py:786-812): a few hundred clauses of a few words,
// a few nodes per graph, whatever edges they have.
//
// On tiles such a data set takes a launch per stage and layer - clauses compiled and ordered, layer 0, hypervector bits
// listed, messages sent, carried and packed, the next layer - each of a few workgroups that live for less time than the
// launch takes, and the tiles have to be made first.  Here a lane is a node: its literal words, then what it received, stay in
// registers; a workgroup's 64 slots hold whole graphs, its waves share the clauses out, and a clause is a handful of
// broadcast LDS reads of include words that all lanes test at once.  What a node sends is gathered in LDS per slot, carried along
// the edges a message word per wave (kernels.py:565-588), and read back.  Bound by its latency: node counts, then literal words, then the
// layers with a barrier or three each: 9 us for 10,000 pairs and 10 clauses of two layers, where the launches on tiles came to 56.
// A call that returns the sums to the host: 85 -> 47 us; two batches of 16 new pairs 364 -> 199.
#pragma once

constexpr int SCORE_SMALL_WAVES = 8;
constexpr int SCORE_SMALL_NODES = 8;     // of the largest graph
constexpr int SCORE_SMALL_VOTES = 4;     // classes that a lane counts for its graph
constexpr int SCORE_SMALL_SLOTS = 16;    // slots of a graph, to have lanes for its classes
constexpr int SCORE_SMALL_QUADS = 2;     // 128-bit reads of literal words, and of message words of one sign
constexpr size_t SCORE_SMALL_LDS = 64 * 1024;
// Where the kernel is the faster way also for clauses that hold at few nodes, which on tiles cost little beyond the launches.
// A workgroup's time grows with its clauses, the quads that it tests of each and the turns in which its lanes count votes, and about
// a thousand workgroups run at once; on tiles a clause takes 2,048 nodes at a time and its included literals only.  us per call on
// a resident data set, here and on tiles, clauses of ten random literals (those of one literal hold at more nodes, where tiles
// take up to five times as long):
//   depth 1, one launch on tiles, too.  20,000 nodes: 10 clauses 31 and 35, 200 clauses of one quad 41 and 42, of two 45
//   and 42, 1,000 clauses 90 and 83; 200,000 nodes: 10 clauses 45 and 35, 200 clauses 96 and 45.
//   message layers.  Graphs of four and eight nodes, 20,000 nodes, 200 clauses, two layers of 256 bits (560,000) 69 and 94;
//   200,000 nodes, 10 clauses 50 and 61, 65 and 52, 200 clauses (1.9 million) 133 and 100.  Two nodes, 200,000 in all: 10 clauses
//   49 and 77, 50 clauses 67 and 84, 200 clauses (1.9 million) 132 and 109; 800,000, two layers, 10 clauses (1.1 million) 151 and 265.
//   Single nodes, 200,000, 200 clauses (2.5 million) 136 and 333; 800,000, 50 clauses (2.5 million) 172 and 722.
constexpr int64_t SCORE_SMALL_GROUPS = 640, SCORE_SMALL_CLAUSE_QUADS = 200;  // depth 1: workgroups, clauses times quads
constexpr int64_t SCORE_SMALL_LAYER_GROUPS = 1300;                           // message layers, more than two nodes: workgroups
// ... for single nodes, two, more: workgroups times clauses times (quads + turns of votes after the first)
constexpr int64_t SCORE_SMALL_TESTED[3] = {2500000, 1250000, 750000};

struct ScoreSmallParams {
    const uint32_t *X, *node_type, *node_index, *n_nodes, *n_edges, *edge_index, *edge;  // n_edges NULL: no edges
    const uint32_t *bank[GTM_MAX_DEPTH];
    const int32_t *weights;
    const uint32_t *hv;
    int32_t *class_sum;
    int first, n_graphs, depth, C, LA, MW, M, MB, B, K, n_types;
    int slots, graphs;  // slots of a graph, graphs of a workgroup
    uint32_t filter;
};

// Include words of a clause in LDS: literal words, then per layer the positive and the negated message words, whole quads each.
__host__ __device__ inline int score_small_stride(int depth, int literal_quads, int message_quads) {
    return 4 * literal_quads + (depth - 1) * 8 * message_quads;
}
inline size_t score_small_lds_words(int C, int K, int MB, int depth, int literal_quads, int message_quads, int graphs) {
    return (size_t)C * score_small_stride(depth, literal_quads, message_quads) + (depth > 1 ? 2 * 4 * message_quads * 64 : 0) +
           (size_t)graphs * K + (size_t)C * (K + (depth > 1 ? MB + 2 : 0));
}

// XQ, MQ: quads of literal words and of message words of one sign.
template <int XQ, int MQ>
__global__ __launch_bounds__(64 * SCORE_SMALL_WAVES) void k_score_small(ScoreSmallParams p) {
    extern __shared__ __align__(16) uint32_t lds[];
    constexpr int THREADS = 64 * SCORE_SMALL_WAVES, XW = 4 * XQ, MWQ = 4 * MQ;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int C = p.C, K = p.K, LA = p.LA, MW = p.MW, MB = p.MB, B = p.B, depth = p.depth;
    const int stride = score_small_stride(depth, XQ, MQ);
    const bool layers = depth > 1;

    uint32_t *inc = lds;                                          // [C][stride]
    uint32_t *sent = inc + (size_t)C * stride;                    // [MWQ][64] what the slots send
    uint32_t *got = sent + (layers ? MWQ * 64 : 0);               // [MWQ][64] ... and receive
    int32_t *sums = (int32_t *)(got + (layers ? MWQ * 64 : 0));   // [graphs][K]
    int32_t *wts = sums + p.graphs * K;                           // [C][K]
    uint32_t *hv = (uint32_t *)(wts + C * K);                     // [C][MB] bits of a message
    uint32_t *truth = hv + C * MB;                                // [C][2] slots at which a clause holds (layers)

    // the lane's slot
    const int gj = lane / p.slots, at = lane - gj * p.slots, first_graph = (int)blockIdx.x * p.graphs;
    const bool has_graph = gj < p.graphs && first_graph + gj < p.n_graphs;
    const int graph = p.first + (has_graph ? first_graph + gj : 0);
    const int n = has_graph ? (int)p.n_nodes[graph] : 0;
    const bool here = at < n && at < p.slots, empty = has_graph && n == 0;
    const int64_t node = here ? (int64_t)p.node_index[graph] + at : 0;
    uint32_t x[XW] = {};
    uint32_t type = 0xFFFFFFFFu, degree = 0u, first_edge = 0u;
    if (here) {
        type = p.node_type[node];
        if (p.n_edges != nullptr && layers) degree = p.n_edges[node], first_edge = p.edge_index[node];
#pragma unroll
        for (int w = 0; w < XW; ++w)
            if (w < LA) x[w] = p.X[node * LA + w];
    }
    // the model: a wave brings the clauses that it will test, a lane per word
    for (int w = lane; w < stride; w += 64) {
        const int in_layers = w - XW, l = in_layers < 0 ? 0 : in_layers / (2 * MWQ) + 1, r = in_layers < 0 ? w : in_layers % (2 * MWQ);
        const int wl = l == 0 ? r : (r < MWQ ? r : MW + r - MWQ), words = l == 0 ? LA : 2 * MW;
        const bool there = l == 0 ? r < LA : (r < MWQ ? r : r - MWQ) < MW;
        const uint32_t *bank = p.bank[0];
#pragma unroll
        for (int b = 1; b < GTM_MAX_DEPTH; ++b)
            if (b == l) bank = p.bank[b];
        const uint32_t keep = !there ? 0u : (l == 0 && wl == LA - 1 ? p.filter : 0xFFFFFFFFu);
        const uint32_t *from = bank + ((int64_t)(there ? wl : 0) * B + (B - 1));
#pragma unroll 4
        for (int c = wave; c < C; c += SCORE_SMALL_WAVES) inc[c * stride + w] = from[(int64_t)c * words * B] & keep;
    }
    for (int k = lane; k < K; k += 64)
        for (int c = wave; c < C; c += SCORE_SMALL_WAVES) wts[c * K + k] = p.weights[(int64_t)k * C + c];
    for (int i = tid; i < p.graphs * K; i += THREADS) sums[i] = 0;
    if (layers) {
        for (int i = tid; i < 2 * MWQ * 64; i += THREADS) sent[i] = 0u;  // (and got)
        for (int i = tid; i < C * MB; i += THREADS) hv[i] = p.hv[i] % (uint32_t)p.M;
    }
    __syncthreads();

    const unsigned long long graph_slots = (p.slots == 64 ? ~0ull : (1ull << p.slots) - 1ull) << (gj * p.slots < 64 ? gj * p.slots : 0);
    int32_t votes[SCORE_SMALL_VOTES] = {};
    const int class_turns = (K + p.slots - 1) / p.slots;
    const int type_step = SCORE_SMALL_WAVES % p.n_types;
    for (int l = 0; l < depth; ++l) {
        uint32_t m[MWQ] = {};
        if (l > 0) {
            __syncthreads();  // everything sent is in LDS
            for (int w = wave; w < MW; w += SCORE_SMALL_WAVES)
                for (uint32_t e = 0; e < degree; ++e) {
                    const uint2 to = reinterpret_cast<const uint2 *>(p.edge)[(int64_t)first_edge + e];
                    const uint32_t turn = to.y < (uint32_t)p.M ? to.y : to.y % (uint32_t)p.M;
                    int from = w - (int)(turn >> 5);
                    if (from < 0) from += MW;
                    const int below = from == 0 ? MW - 1 : from - 1;
                    const unsigned long long both = (unsigned long long)sent[from * 64 + lane] << 32 | sent[below * 64 + lane];
                    const uint32_t v = (uint32_t)((both << (turn & 31u)) >> 32);
                    if (v != 0u && to.x < (uint32_t)n) atomicOr(&got[w * 64 + gj * p.slots + (int)to.x], v);
                }
            __syncthreads();
#pragma unroll
            for (int w = 0; w < MWQ; ++w)
                if (w < MW) m[w] = got[w * 64 + lane];
            if (l + 1 < depth) {
                __syncthreads();  // everything received is in registers
                for (int i = tid; i < 2 * MWQ * 64; i += THREADS) sent[i] = 0u;
                __syncthreads();
            }
        }
        int clause_type = wave % p.n_types;
        for (int c = wave; c < C; c += SCORE_SMALL_WAVES) {
            bool holds;
            if (l == 0) {
                const uint4 *words = reinterpret_cast<const uint4 *>(inc + c * stride);
                uint32_t bad = 0u;
#pragma unroll
                for (int q = 0; q < XQ; ++q) {
                    const uint4 i = words[q];
                    bad |= (i.x & ~x[4 * q]) | (i.y & ~x[4 * q + 1]) | (i.z & ~x[4 * q + 2]) | (i.w & ~x[4 * q + 3]);
                }
                holds = bad == 0u && type == (uint32_t)clause_type;
                clause_type += type_step;
                if (clause_type >= p.n_types) clause_type -= p.n_types;
            } else {
                const uint4 *words = reinterpret_cast<const uint4 *>(inc + c * stride + XW + (l - 1) * 2 * MWQ);
                uint32_t bad = 0u;
#pragma unroll
                for (int q = 0; q < MQ; ++q) {
                    const uint4 i = words[q], j = words[MQ + q];
                    bad |= (i.x & ~m[4 * q]) | (i.y & ~m[4 * q + 1]) | (i.z & ~m[4 * q + 2]) | (i.w & ~m[4 * q + 3]);
                    bad |= (j.x & m[4 * q]) | (j.y & m[4 * q + 1]) | (j.z & m[4 * q + 2]) | (j.w & m[4 * q + 3]);
                }
                holds = bad == 0u && ((truth[2 * c + (lane >> 5)] >> (lane & 31)) & 1u);
            }
            const unsigned long long all = __ballot(holds);
            if (l + 1 < depth) {
                if (lane < 2) truth[2 * c + lane] = (uint32_t)(all >> (32 * lane));  // (read by this wave alone)
                if (holds)
                    for (int j = 0; j < MB; ++j) {
                        const uint32_t bit = hv[c * MB + j];
                        atomicOr(&sent[(bit >> 5) * 64 + lane], 1u << (bit & 31u));
                    }
            } else {
                // (the reference's arithmetic has every clause vote for a graph without nodes, kernels.py:289-295)
                const bool fired = (all & graph_slots) != 0ull || empty;
#pragma unroll
                for (int u = 0; u < SCORE_SMALL_VOTES; ++u)
                    if (u < class_turns) {
                        const int k = at + u * p.slots;
                        const int32_t weight = wts[c * K + (k < K ? k : 0)];
                        votes[u] += fired ? weight : 0;
                    }
            }
        }
    }
    if (has_graph)
#pragma unroll
        for (int u = 0; u < SCORE_SMALL_VOTES; ++u)
            if (at + u * p.slots < K && votes[u] != 0) atomicAdd(&sums[gj * K + at + u * p.slots], votes[u]);
    __syncthreads();
    const int results = min(p.graphs, p.n_graphs - first_graph) * K;
    for (int i = tid; i < results; i += THREADS) p.class_sum[(int64_t)first_graph * K + i] = sums[i];
}
