// Building the literal-major tiles of a data set (layout: score_tiles.h) from its node-major
// literal words, once per data set and tile geometry.
//
// A wave takes 256 node slots (8 words of the tile's rows) and one quad of literal words: a lane loads
// 16 bytes of its slot's node, four times, and 32 x 32 bit transpositions across the lanes of each
// half-wave turn them into 4 words of 128 rows, stored 16 bytes per lane.  Every literal word is read
// once and every tile word written once, so what bounds the kernel is memory; what it must avoid is
// reading a bit at a time, as one thread per tile word did (32 words of 32 nodes for ONE word of a row).
// The waves of a workgroup take the quads of the same slots together, so that the pieces of a node's row
// and of a tile row that they touch meet in the L2.  The number of nodes at which each literal holds falls
// out of the words at hand and is added up in LDS, then once per row and workgroup in memory.
//
// Measured, 10,000 images of 361 nodes and 8 literal words (115 MB in, 126 + 63 MB out): 97 us, where the thread
// per tile word and the passes for the counts and for `xpos` took 2,870 + 97 + 34 us; 1,000 grids of 841 nodes and 64
// literal words (215 MB in, 230 MB out): 190 us (4,000 + 600); 10,000 images of one node and 128 words: 15 us (218).
#pragma once

constexpr int TILE_BUILD_BLOCK = 1024;
constexpr int TILE_BUILD_WORDS = 8;   // words of a tile row per task of a wave
constexpr int TILE_BUILD_QUADS = 64;  // most quads of literal words a workgroup counts in LDS (32 KB)

struct TileBuildShape {
    int quads;        // quads of literal words
    int word_groups;  // groups of TILE_BUILD_WORDS words of a row
    int quad_parts, quads_per_part;    // a tile's quads, and its word groups, are shared out among
    int word_parts, groups_per_part;   // quad_parts x word_parts workgroups
    unsigned tile_blocks;              // workgroups in the tiles' direction; each takes every tile_blocks-th tile
};

// Few tiles: a tile's literals, then its words, are shared out until there are about two workgroups per CU (at
// least one task per wave of each).  Many tiles: at most 1,024 workgroups, each for several tiles, because every
// workgroup adds its counts to the same words of memory, one after the other (about 30 ns each).
inline TileBuildShape tile_build_shape(const TileGeom &tg, int LA) {
    TileBuildShape s{};
    s.quads = (LA + 3) / 4;
    s.word_groups = (tg.tw + TILE_BUILD_WORDS - 1) / TILE_BUILD_WORDS;
    const int wanted = tg.n_tiles < 512 ? (512 + tg.n_tiles - 1) / tg.n_tiles : 1;
    auto parts_of = [](int items, int parts, int least) {
        const int most = items / least > 1 ? items / least : 1;
        return parts < most ? parts : most;
    };
    constexpr int WAVES = TILE_BUILD_BLOCK / 64;
    s.quad_parts = parts_of(s.quads, wanted, s.word_groups >= WAVES ? 1 : (WAVES + s.word_groups - 1) / s.word_groups);
    s.quads_per_part = (s.quads + s.quad_parts - 1) / s.quad_parts;
    if (s.quads_per_part > TILE_BUILD_QUADS) s.quads_per_part = TILE_BUILD_QUADS;
    s.quad_parts = (s.quads + s.quads_per_part - 1) / s.quads_per_part;
    s.word_parts = parts_of(s.word_groups, (wanted + s.quad_parts - 1) / s.quad_parts,
                            (WAVES + s.quads_per_part - 1) / s.quads_per_part);
    s.groups_per_part = (s.word_groups + s.word_parts - 1) / s.word_parts;
    s.word_parts = (s.word_groups + s.groups_per_part - 1) / s.groups_per_part;
    s.tile_blocks = (unsigned)(tg.n_tiles < 1024 ? tg.n_tiles : 1024);
    return s;
}

// LDS words: a count per row of the part's literals.
inline size_t tile_build_lds_words(const TileBuildShape &s) { return (size_t)s.quads_per_part * 128; }

// grid (tile_blocks, quad_parts, word_parts).  row_count[rows] is zero on entry and filled for the literals' rows.  ALIGNED: LA is a multiple of 4, so a
// quad of a node's literal words is one 16-byte load.
template <bool ALIGNED>
__global__ __launch_bounds__(TILE_BUILD_BLOCK) void k_build_tiles(
    const uint32_t *__restrict__ X, const uint32_t *__restrict__ node_type, const uint32_t *__restrict__ node_index,
    const uint32_t *__restrict__ n_nodes_arr, int G, int LA, int literals, int n_types, TileGeom tg, TileBuildShape s,
    uint32_t *__restrict__ tiles, unsigned long long *row_count, uint32_t *__restrict__ xpos) {
    extern __shared__ uint32_t counts[];  // [quads of the part * 128]
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, bit = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr int WAVES = TILE_BUILD_BLOCK / 64;
    const int q0 = blockIdx.y * s.quads_per_part, n_quads = min(s.quads_per_part, s.quads - q0);
    const int g0 = blockIdx.z * s.groups_per_part, n_groups = min(s.groups_per_part, s.word_groups - g0);
    const bool with_types = blockIdx.y == 0;  // the node-type rows and the all-ones row go with the first quads
    for (int i = tid; i < s.quads_per_part * 128; i += TILE_BUILD_BLOCK) counts[i] = 0u;
    __syncthreads();
    const int kinds = n_quads + (with_types ? 1 : 0);  // tasks per word group
    const int pos_words = literals / 64;               // words of a node's positive literals (half tiles)
    for (int tile = blockIdx.x; tile < tg.n_tiles; tile += gridDim.x) {
        uint32_t *out = tiles + (int64_t)tile * tg.rows * tg.tw;
        for (int t = wave; t < n_groups * kinds; t += WAVES) {
            const int wg = t / kinds, q = q0 + (t - wg * kinds);
            const bool types_task = t - wg * kinds == n_quads;
            const int w0 = (g0 + wg) * TILE_BUILD_WORDS + 4 * half;  // this half-wave's 4 words of every row
            const bool words_exist = w0 < tg.tw;                       // (tw is a multiple of 4)
            // the nodes in this lane's 4 slots; a graph without nodes has every bit of its first slot set: the
            // reference's chunk arithmetic leaves every clause true for it (kernels.py:289-295, 443-466)
            int64_t node[4];
            uint32_t stand_in[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int pos = (w0 + k) * 32 + bit, j = pos / tg.slot_bits, n = pos - j * tg.slot_bits;
                const int64_t g = (int64_t)tile * tg.gpt + j;
                const bool graph = words_exist && j < tg.gpt && g < G;
                const uint32_t count = graph ? n_nodes_arr[g] : 1u;
                node[k] = graph && (uint32_t)n < count ? (int64_t)node_index[g] + n : -1;
                stand_in[k] = count == 0u && n == 0 ? 0xFFFFFFFFu : 0u;
            }
            if (types_task) {
                uint32_t type[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) type[k] = node[k] >= 0 ? node_type[node[k]] : 0xFFFFFFFFu;
                for (int ty = 0; ty < n_types; ++ty) {
                    uint32_t word[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const unsigned long long m = __ballot((node[k] >= 0 && type[k] == (uint32_t)ty) || stand_in[k] != 0u);
                        word[k] = half ? (uint32_t)(m >> 32) : (uint32_t)m;
                    }
                    if (bit == 0 && words_exist)
                        *(uint4 *)(out + (int64_t)(literals + ty) * tg.tw + w0) = make_uint4(word[0], word[1], word[2], word[3]);
                }
                if (bit == 0 && words_exist) {
                    // all ones over the graph slots; words that only pad the row stay 0 so that they never keep a
                    // clause alive
                    const int used = tg.slot_words == 0 ? tg.tw : tg.gpt * tg.slot_words;
                    uint32_t word[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) word[k] = w0 + k < used ? 0xFFFFFFFFu : 0u;
                    *(uint4 *)(out + (int64_t)(tg.rows - 1) * tg.tw + w0) = make_uint4(word[0], word[1], word[2], word[3]);
                }
                continue;
            }
            uint32_t v[4][4];  // [slot word][literal word of the quad]
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const uint32_t *row = X + node[k] * LA + 4 * q;
                if constexpr (ALIGNED) {
                    const uint4 x = node[k] >= 0 ? *(const uint4 *)row : make_uint4(0u, 0u, 0u, 0u);
                    v[k][0] = x.x, v[k][1] = x.y, v[k][2] = x.z, v[k][3] = x.w;
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[k][i] = node[k] >= 0 && 4 * q + i < LA ? row[i] : 0u;
                }
            }
            if (xpos && words_exist) {
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    uint32_t *to = xpos + ((int64_t)tile * tg.tw * 32 + (w0 + k) * 32 + bit) * pos_words + 4 * q;
                    if (pos_words % 4 == 0 && 4 * q < pos_words)
                        *(uint4 *)to = make_uint4(v[k][0], v[k][1], v[k][2], v[k][3]);
                    else
                        for (int i = 0; i < 4 && 4 * q + i < pos_words; ++i) to[i] = v[k][i];
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                uint32_t word[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) word[k] = tile_transpose32(v[k][i] | stand_in[k], lane);
                const int row = (4 * q + i) * 32 + bit;
                if (row < literals && words_exist) {
                    *(uint4 *)(out + (int64_t)row * tg.tw + w0) = make_uint4(word[0], word[1], word[2], word[3]);
                    const uint32_t held = __popc(word[0]) + __popc(word[1]) + __popc(word[2]) + __popc(word[3]);
                    if (held) atomicAdd(&counts[row - q0 * 128], held);
                }
            }
        }
    }
    __syncthreads();
    for (int i = tid; i < n_quads * 128; i += TILE_BUILD_BLOCK)
        if (counts[i]) atomicAdd(&row_count[q0 * 128 + i], (unsigned long long)counts[i]);
}

// Literal rows ordered by how often they hold in the data set, rarest first: order[r] = literal with rank r under
// the key (row_count, literal).  A wave ranks TILE_ORDER_AT_ONCE literals: its lanes go over all keys, 64 at a time,
// and count those below each - work for the whole chip, where one thread per literal going over all keys by itself
// took 280 us for 4,096 literals (16 workgroups, one load at a time): 25 us.
constexpr int TILE_ORDER_AT_ONCE = 4;

__global__ __launch_bounds__(256) void k_row_order(const unsigned long long *__restrict__ row_count, int literals,
                                                   uint32_t *__restrict__ order) {
    const int lane = threadIdx.x & 63;
    const int first = (int)(blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * TILE_ORDER_AT_ONCE;
    if (first >= literals) return;
    unsigned long long mine[TILE_ORDER_AT_ONCE];
    int rank[TILE_ORDER_AT_ONCE];
#pragma unroll
    for (int u = 0; u < TILE_ORDER_AT_ONCE; ++u) {
        mine[u] = row_count[min(first + u, literals - 1)];
        rank[u] = 0;
    }
    for (int m = lane; m < literals; m += 64) {
        const unsigned long long other = row_count[m];
#pragma unroll
        for (int u = 0; u < TILE_ORDER_AT_ONCE; ++u) rank[u] += (other < mine[u]) || (other == mine[u] && m < first + u);
    }
#pragma unroll
    for (int u = 0; u < TILE_ORDER_AT_ONCE; ++u) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) rank[u] += __shfl_xor(rank[u], off);
        if (lane == 0 && first + u < literals) order[rank[u]] = (uint32_t)(first + u);
    }
}
