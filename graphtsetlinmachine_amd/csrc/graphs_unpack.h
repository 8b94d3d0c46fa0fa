// The arrays of a data set as the kernels index them, from the packed form that came over the bus (pack.c): the
// negated literals as complements of the positive ones, small numbers widened, a node's first edge by a running
// sum over the edge counts of its graph.
//
// One launch; its workgroups are shared out among the words of X, the nodes, the graphs and the edges.  A thread
// writes one word after the other of its array, neighbouring threads neighbouring words, so the kernel is bound by
// memory, and small beside the bus.  Scoring 999 new images (12.8 MB of literal words and 4.3 MB of indexes, of which
// 6.4 MB are sent): 920 -> 395 us per batch; first pass over 1,000 grids (215 MB): 13.9 -> 7.5 ms.
#pragma once

constexpr int UNPACK_BLOCK = 256;
constexpr int UNPACK_WORDS = 8;  // words of X, or numbers of `edge`, per thread

struct UnpackShape {
    unsigned row_blocks, node_blocks, graph_blocks, edge_blocks;
};

__device__ __forceinline__ uint32_t unpack_number(const void *in, int64_t i, int bytes, uint32_t value) {
    return bytes == 0 ? value : bytes == 1 ? ((const uint8_t *)in)[i] : bytes == 2 ? ((const uint16_t *)in)[i] : ((const uint32_t *)in)[i];
}

__global__ __launch_bounds__(UNPACK_BLOCK) void k_unpack_graphs(gtm_packed_graphs p, UnpackShape s) {
    unsigned block = blockIdx.x;
    const int tid = threadIdx.x;
    if (block < s.row_blocks) {
        const int64_t total = p.total_nodes * p.literal_words;
        const int64_t base = (int64_t)block * (UNPACK_BLOCK * UNPACK_WORDS) + tid;
        if (!p.rows_positive) {
#pragma unroll
            for (int u = 0; u < UNPACK_WORDS; ++u) {
                const int64_t i = base + u * UNPACK_BLOCK;
                if (i < total) p.X[i] = p.rows[i];
            }
            return;
        }
        const int hv = p.hypervector_size, words = (hv + 31) / 32, LA = p.literal_words;
        const uint32_t last = hv % 32 == 0 ? 0xFFFFFFFFu : (1u << (hv % 32)) - 1u;
        // (one 64-bit division per workgroup; a thread's own, from the workgroup's first node on, are short)
        const int64_t block_base = base - tid, node0 = block_base / LA;
        const uint32_t into = (uint32_t)(block_base - node0 * LA) + (uint32_t)tid;
#pragma unroll
        for (int u = 0; u < UNPACK_WORDS; ++u) {
            const int64_t i = base + u * UNPACK_BLOCK;
            if (i >= total) break;
            const uint32_t at = into + u * UNPACK_BLOCK, ahead = at / (uint32_t)LA;
            const int w = (int)(at - ahead * (uint32_t)LA);
            const uint32_t *row = p.rows + (node0 + ahead) * words;
            uint32_t out = w < words ? row[w] : 0u;
            // bit 32 w + b of the row is the complement of positive bit 32 w + b - hv
            const int from = w * 32 - hv;
            auto negated = [&](int word) { return word < 0 || word >= words ? 0u : ~row[word] & (word == words - 1 ? last : 0xFFFFFFFFu); };
            if (from > -32) {
                const int low = from >= 0 ? from >> 5 : -1, shift = from & 31;
                out |= negated(low) >> shift;
                if (shift) out |= negated(low + 1) << (32 - shift);
            }
            p.X[i] = out;
        }
        return;
    }
    block -= s.row_blocks;
    if (block < s.node_blocks) {
        const int64_t i = (int64_t)block * UNPACK_BLOCK + tid;
        if (i < p.total_nodes) {
            p.node_type[i] = unpack_number(p.types, i, p.type_bytes, p.type_value);
            p.number_of_graph_node_edges[i] = unpack_number(p.degrees, i, p.degree_bytes, p.degree_value);
            if (!p.index_follows) p.edge_index[i] = p.first_edges[i];
        }
        if (i < p.number_of_graphs) {
            p.node_index[i] = p.first_nodes[i];
            p.number_of_graph_nodes[i] = p.node_counts[i];
        }
        return;
    }
    block -= s.node_blocks;
    if (block < s.graph_blocks) {
        // a wave per graph: running sum of the edge counts, 64 nodes at a time
        const int lane = tid & 63;
        const int64_t g = (int64_t)block * (UNPACK_BLOCK / 64) + (tid >> 6);
        if (g >= p.number_of_graphs) return;
        const int64_t first = p.first_nodes[g];
        const int n = (int)p.node_counts[g];
        uint32_t before = p.first_edges[g];
        for (int n0 = 0; n0 < n; n0 += 64) {
            const uint32_t own = n0 + lane < n ? unpack_number(p.degrees, first + n0 + lane, p.degree_bytes, p.degree_value) : 0u;
            uint32_t sum = own;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const uint32_t v = (uint32_t)__shfl_up((int)sum, off);
                if (lane >= off) sum += v;
            }
            if (n0 + lane < n) p.edge_index[first + n0 + lane] = before + sum - own;
            before += (uint32_t)__shfl((int)sum, 63);
        }
        return;
    }
    block -= s.graph_blocks;
    const int64_t base = (int64_t)block * (UNPACK_BLOCK * UNPACK_WORDS) + tid;
#pragma unroll
    for (int u = 0; u < UNPACK_WORDS; ++u) {
        const int64_t i = base + u * UNPACK_BLOCK;
        if (i < 2 * p.total_edges) p.edge[i] = unpack_number(p.edges, i, p.edge_bytes, 0u);
    }
}
