// The message rows of a layer when a data set's edges are a few MOVES.
//
// An edge goes from node n to node n + d and has a type t.  In chains, grids and pairs - nodes numbered in
// the order of what they stand for - only a few (t, d) occur in the whole data set: 'Right' is +1, 'Up' is one
// row of the grid.  What the nodes receive (kernels.py:565-588) then needs no vector per node, no walk along
// edges and no transposition, in either direction: received row p of a tile is the OR over the moves of the SENT
// row (p - t) mod M shifted by d bits, kept where such an edge ends.
//
// k_edge_moves finds the (t, d) of a data set, k_edge_move_masks the slots where each of them ends; both run once
// per data set (gtm_build_moves).  A data set with more than TILE_MOVES_MAX of them, with a type or an offset too
// large for a key, or with an edge that leaves its graph, keeps the kernels that walk the edges.
// Measured, whole scoring passes, edges walked -> rows shifted: 3,000 chains of 1,000 nodes (messages of 512 bits) 481 ->
// 318 us, 1,000 grids of 841 nodes (two layers of 1,024 bits, 8,000 clauses) 2,890 -> 2,593, 10,000 pairs 111 -> 86;
// transform of 4,001 chains of 3 to 41 nodes, three layers deep, 772 -> 569.
#pragma once

constexpr int TILE_MOVES_MAX = 8;
constexpr int TILE_MOVES_HEADER_WORDS = 16;  // TILE_MOVES_MAX keys (0: none), then != 0 when the moves do not describe the edges
constexpr int TILE_MOVES_BLOCK = 256;

// What a message kernel is told, worked out on the host from the keys.
struct TileMoves {
    int n;                            // 0: the edges are walked
    int type[TILE_MOVES_MAX];
    int words[TILE_MOVES_MAX];        // slot s receives from slot s + 32 words + bits, 0 <= bits < 32
    int bits[TILE_MOVES_MAX];
};

constexpr uint32_t TILE_MOVE_OFFSET = 1u << 15, TILE_MOVE_TYPES = 1u << 15;

// 0 when the edge is no move.
__device__ __forceinline__ uint32_t tile_move_key(uint32_t from, uint32_t to, uint32_t type, uint32_t n) {
    const uint32_t d = to - from + TILE_MOVE_OFFSET;  // (nodes of a tile's graph are far fewer than 2^15)
    return to < n && type < TILE_MOVE_TYPES && d - 1u < 2u * TILE_MOVE_OFFSET - 1u ? (type << 16) | d : 0u;
}

// A key into a workgroup's table in LDS, where it is not there yet; false: it is no key, or there is no room.
__device__ __forceinline__ bool tile_move_noted(uint32_t *keys, uint32_t key) {
    if (key == 0u) return false;
    for (int k = 0; k < TILE_MOVES_MAX; ++k) {
        uint32_t held = *(volatile uint32_t *)&keys[k];
        if (held == 0u) held = atomicCAS(&keys[k], 0u, key);
        if (held == key || held == 0u) return true;
    }
    return false;
}
// A workgroup's table -> the header in memory (one thread).
__device__ __forceinline__ void tile_moves_publish(const uint32_t *keys, uint32_t lost, uint32_t *header) {
    for (int j = 0; j < TILE_MOVES_MAX && keys[j] && !lost; ++j) {
        int k = 0;
        for (; k < TILE_MOVES_MAX; ++k) {
            uint32_t held = __hip_atomic_load(&header[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (held == 0u) held = atomicCAS(&header[k], 0u, keys[j]);
            if (held == keys[j] || held == 0u) break;
        }
        if (k == TILE_MOVES_MAX) lost = 1u;
    }
    if (lost) atomicOr(&header[TILE_MOVES_MAX], 1u);
}

// The node in slot `pos` of a tile: its place in the data set's node arrays, its number in its graph and the graph's
// nodes and first slot; false when there is none.
__device__ __forceinline__ bool tile_slot_node(const TileGeom &tg, int tile, int pos, int G, const uint32_t *node_index,
                                               const uint32_t *n_nodes, int64_t *row, uint32_t *n, uint32_t *nodes, int *slot0) {
    const int j = pos / tg.slot_bits;
    const int64_t g = (int64_t)tile * tg.gpt + j;
    if (j >= tg.gpt || g >= G) return false;
    *slot0 = j * tg.slot_bits;
    *n = (uint32_t)(pos - *slot0);
    *nodes = n_nodes[g];
    if (*n >= *nodes) return false;
    *row = (int64_t)node_index[g] + *n;
    return true;
}

// The keys of a data set's edges -> header (zero on entry).  A workgroup collects the keys of its slots in LDS and
// adds those that it has not seen in memory to the table there: few atomics whatever the number of edges.  Bound
// by reading the edges: 3,000 chains of 1,000 nodes, 48 MB of edges and 36 MB of node arrays.
__global__ __launch_bounds__(TILE_MOVES_BLOCK) void k_edge_moves(TileGeom tg, int G, const uint32_t *__restrict__ node_index,
                                                                  const uint32_t *__restrict__ n_nodes,
                                                                  const uint32_t *__restrict__ n_edges,
                                                                  const uint32_t *__restrict__ edge_index,
                                                                  const uint32_t *__restrict__ edge, uint32_t *header) {
    __shared__ uint32_t keys[TILE_MOVES_MAX], too_many;
    if (threadIdx.x < TILE_MOVES_MAX) keys[threadIdx.x] = 0u;
    if (threadIdx.x == 0) too_many = 0u;
    __syncthreads();
    const int64_t slots = (int64_t)tg.n_tiles * tg.tw * 32;
    for (int64_t s = (int64_t)blockIdx.x * TILE_MOVES_BLOCK + threadIdx.x; s < slots; s += (int64_t)gridDim.x * TILE_MOVES_BLOCK) {
        const int tile = (int)(s / (tg.tw * 32)), pos = (int)(s - (int64_t)tile * tg.tw * 32);
        int64_t row;
        uint32_t n, nodes;
        int slot0;
        if (!tile_slot_node(tg, tile, pos, G, node_index, n_nodes, &row, &n, &nodes, &slot0)) continue;
        const uint32_t count = n_edges[row];
        const uint2 *out_edges = reinterpret_cast<const uint2 *>(edge) + edge_index[row];
        for (uint32_t e = 0; e < count; ++e) {
            if (*(volatile uint32_t *)&too_many) break;
            const uint2 to = out_edges[e];
            if (!tile_move_noted(keys, tile_move_key(n, to.x, to.y, nodes))) too_many = 1u;
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) tile_moves_publish(keys, too_many, header);
}

// masks[tile][move][tw]: the slots where an edge of the move ends.  One workgroup per tile at a time; nothing when
// the table above overflowed.
__global__ __launch_bounds__(TILE_MOVES_BLOCK) void k_edge_move_masks(TileGeom tg, int G, const uint32_t *__restrict__ node_index,
                                                                       const uint32_t *__restrict__ n_nodes,
                                                                       const uint32_t *__restrict__ n_edges,
                                                                       const uint32_t *__restrict__ edge_index,
                                                                       const uint32_t *__restrict__ edge,
                                                                       const uint32_t *__restrict__ header, uint32_t *__restrict__ masks) {
    extern __shared__ uint32_t ends[];  // [TILE_MOVES_MAX][tw]
    if (header[TILE_MOVES_MAX]) return;
    uint32_t keys[TILE_MOVES_MAX];
#pragma unroll
    for (int k = 0; k < TILE_MOVES_MAX; ++k) keys[k] = header[k];
    const int words = TILE_MOVES_MAX * tg.tw;
    for (int tile = blockIdx.x; tile < tg.n_tiles; tile += gridDim.x) {
        for (int i = threadIdx.x; i < words; i += TILE_MOVES_BLOCK) ends[i] = 0u;
        __syncthreads();
        for (int pos = threadIdx.x; pos < tg.tw * 32; pos += TILE_MOVES_BLOCK) {
            int64_t row;
            uint32_t n, nodes;
            int slot0;
            if (!tile_slot_node(tg, tile, pos, G, node_index, n_nodes, &row, &n, &nodes, &slot0)) continue;
            const uint32_t count = n_edges[row];
            const uint2 *out_edges = reinterpret_cast<const uint2 *>(edge) + edge_index[row];
            for (uint32_t e = 0; e < count; ++e) {
                const uint2 to = out_edges[e];
                const uint32_t key = tile_move_key(n, to.x, to.y, nodes);
                const int slot = slot0 + (int)to.x;
#pragma unroll
                for (int k = 0; k < TILE_MOVES_MAX; ++k)
                    if (key && key == keys[k]) atomicOr(&ends[k * tg.tw + (slot >> 5)], 1u << (slot & 31));
            }
        }
        __syncthreads();
        for (int i = threadIdx.x; i < words; i += TILE_MOVES_BLOCK) masks[(int64_t)tile * words + i] = ends[i];
        __syncthreads();
    }
}

// LDS words of k_tile_messages_moved: the sent rows between two runs of words that a shifted read may touch (what it
// finds there the masks remove), and the masks.
__host__ __device__ inline int tile_moves_margin(const TileGeom &g) { return g.tw + 8; }
inline size_t tile_messages_moved_lds_words(const TileGeom &g, int M, int n_moves) {
    return (size_t)M * g.tw + 2 * tile_moves_margin(g) + (size_t)n_moves * g.tw;
}

// The four words that start A words into eight.
template <int A>
__device__ __forceinline__ void tile_moved_quad(const uint32_t (&v)[8], int bits, const uint4 &mask, uint32_t (&out)[4]) {
    const uint32_t m[4] = {mask.x, mask.y, mask.z, mask.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) out[i] |= __builtin_amdgcn_alignbit(v[A + i + 1], v[A + i], bits) & m[i];
}

// Workgroup (tile, part): the rows [M + 2][tw] that the next layer's evaluation stages (the part's share of the M).
//   1. sent rows in LDS, literal-major: row p is the OR of the truth rows of the clauses whose hypervector holds
//      bit p.  LISTED: the clauses that the evaluation before listed as alive (rows of at most 64 words, the
//      function of score_messages.h); else all of them, 16 bytes of a row per thread;
//   2. every thread makes four words of a received row from two aligned 16-byte reads per move.
// Few tiles leave CUs idle: then several workgroups share a tile, each with all sent rows and a share of the
// received ones.  FORM 0: every clause; 1, 2: listed clauses, rows of at most 32, 64 words.
template <int FORM>
__global__ __launch_bounds__(TILE_MESSAGES_LDS_BLOCK) void k_tile_messages_moved(
    const uint32_t *__restrict__ bitmap, int C, TileGeom tg, int tile0, int G, int M, const uint32_t *__restrict__ hv, int MB,
    const uint32_t *__restrict__ alive, int streams, int alive_stride, const uint32_t *__restrict__ n_nodes, TileMoves moves,
    const uint32_t *__restrict__ masks, uint32_t *__restrict__ rows) {
    extern __shared__ __align__(16) uint32_t lds[];
    constexpr int NT = TILE_MESSAGES_LDS_BLOCK;
    const int tid = threadIdx.x, tw = tg.tw, quads = tw >> 2, tile_local = blockIdx.x;
    const int margin = tile_moves_margin(tg);
    uint32_t *sent = lds + margin;
    uint4 *ends = reinterpret_cast<uint4 *>(sent + (size_t)M * tw + margin);  // [n][tw]
    uint32_t *out = rows + (int64_t)tile_local * (M + 2) * tw;

    for (int i = tid; i < M * quads; i += NT) reinterpret_cast<uint4 *>(sent)[i] = make_uint4(0u, 0u, 0u, 0u);
    const uint4 *mask_rows = reinterpret_cast<const uint4 *>(masks + (int64_t)(tile0 + tile_local) * TILE_MOVES_MAX * tw);
    for (int i = tid; i < moves.n * quads; i += NT) ends[i] = mask_rows[i];
    __syncthreads();

    // item i of this thread is (row, quad) number tid + i NT: one division, then steps
    const int step_row = NT / quads, step_quad = NT - step_row * quads;
    if constexpr (FORM == 0) {
        const uint4 *truth = reinterpret_cast<const uint4 *>(bitmap + (int64_t)tile_local * C * tw);
        const int total = C * quads;
        int c = tid / quads, q = tid - c * quads;
        for (int at = tid; at < total; at += 4 * NT) {
            uint4 t[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) t[u] = truth[min(at + u * NT, total - 1)];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const unsigned long long lo = ((unsigned long long)t[u].y << 32) | t[u].x, hi = ((unsigned long long)t[u].w << 32) | t[u].z;
                if (at + u * NT < total && (lo | hi) != 0ull)
                    for (int j = 0; j < MB; ++j) {
                        const uint32_t h = hv[(int64_t)c * MB + j];
                        if (h >= (uint32_t)M) continue;
                        unsigned long long *row = reinterpret_cast<unsigned long long *>(sent + h * (uint32_t)tw + 4 * q);
                        if (lo) atomicOr(row, lo);
                        if (hi) atomicOr(row + 1, hi);
                    }
                c += step_row, q += step_quad;
                if (q >= quads) q -= quads, ++c;
            }
        }
    } else {
        tile_sent_rows_listed<FORM == 2>(sent, bitmap, tile_local, C, tw, M, hv, MB, alive, streams, alive_stride);
    }
    __syncthreads();

    const int p_lo = (int)((int64_t)M * blockIdx.y / gridDim.y), p_hi = (int)((int64_t)M * (blockIdx.y + 1) / gridDim.y);
    int row = tid / quads, q = tid - row * quads;
    for (int at = tid; at < (p_hi - p_lo) * quads; at += NT) {
        uint32_t got[4] = {0u, 0u, 0u, 0u};
        for (int k = 0; k < moves.n; ++k) {
            int from = p_lo + row - moves.type[k];
            from += from < 0 ? M : 0;
            const int word = from * tw + 4 * q + (moves.words[k] & ~3);
            const uint4 a = *reinterpret_cast<const uint4 *>(sent + word), b = *reinterpret_cast<const uint4 *>(sent + word + 4);
            const uint4 mask = ends[k * quads + q];
            const uint32_t v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
            switch (moves.words[k] & 3) {  // (the same for every thread)
            case 0: tile_moved_quad<0>(v, moves.bits[k], mask, got); break;
            case 1: tile_moved_quad<1>(v, moves.bits[k], mask, got); break;
            case 2: tile_moved_quad<2>(v, moves.bits[k], mask, got); break;
            default: tile_moved_quad<3>(v, moves.bits[k], mask, got); break;
            }
        }
        reinterpret_cast<uint4 *>(out)[(int64_t)(p_lo + row) * quads + q] = make_uint4(got[0], got[1], got[2], got[3]);
        row += step_row, q += step_quad;
        if (q >= quads) q -= quads, ++row;
    }
    if (blockIdx.y == 0) tile_rows_after_messages(out, tg, tile0 + tile_local, G, M, n_nodes);
}
