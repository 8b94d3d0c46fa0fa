/* A data set's arrays made small for the trip to the device.
 *
 * The bus carries 57 GB/s where the device's memory carries 4,700, and most of what Graphs builds follows from
 * less: a negated literal is the complement of its positive one (graphs.py:148-159), the first edge of a node
 * follows from the edge counts before it (graphs.py:128), and node types, edge counts and edge ends are small
 * numbers.  Whether that holds is looked at word by word while packing - the arrays are public - and what does
 * not hold goes as it is.  gtm_unpack_graphs (gtm_hip.hip) makes the reference's arrays of it on the device.
 *
 * Loops over whole arrays, spread over OpenMP threads from PACK_PARALLEL items on: below that, waking the
 * threads takes longer than the work.
 */
#include <stdint.h>
#include <string.h>

#define PACK_PARALLEL 16384

/* A graph's first edges are summed up by one thread here and by one wave on the device: together 7 ns per node of the
 * largest graph, where sending them costs a node 0.1.  So they follow only where graphs are small (1,024 nodes: 7 us),
 * or the largest is at most a 64th of all nodes and the others are summed beside it.  Upload of one graph of 1,000,000
 * nodes 7.8 ms summed, 0.94 sent (1.2 by plain copies); of four of 100,000 1.16 and 0.47; of one of 20,000 236 and
 * 126 us; a hundred of 10,000 are summed in 0.73 to 0.79 ms (1.26 by plain copies). */
#define PACK_SUMMED 1024
#define PACK_SUMMED_SHARE 64

/* How a data set's small arrays can be sent: the fields of `plan`. */
enum {
    PLAN_TYPE_BYTES,      /* bytes per node type: 0 (all alike), 1 or 4 */
    PLAN_TYPE_VALUE,      /* the type of all nodes where 0 */
    PLAN_DEGREE_BYTES,    /* the same for the number of edges of a node */
    PLAN_DEGREE_VALUE,
    PLAN_INDEX_FOLLOWS,   /* 1: a node's first edge = edge_start of its graph + the edges of the graph's nodes before it */
    PLAN_EDGE_BYTES,      /* bytes per number of `edge`: 2 or 4 */
    PLAN_EMPTY_GRAPH,     /* 1: some graph has no nodes */
};

static uint32_t bytes_for(uint32_t differences, uint32_t all) { return differences == 0 ? 0 : all < 256 ? 1 : 4; }

/* edge_start[G] is filled where PLAN_INDEX_FOLLOWS comes out as 1. */
void gtm_pack_plan(const uint32_t *node_type, const uint32_t *degree, const uint32_t *edge_index, const uint32_t *node_index,
                   const uint32_t *n_nodes, const uint32_t *edge, int64_t N, int64_t E, int64_t G, uint32_t *plan,
                   uint32_t *edge_start) {
    uint32_t type_differs = 0, type_all = 0, degree_differs = 0, degree_all = 0, edge_all = 0, index_bad = 0, empty = 0, largest = 0;
    const uint32_t type0 = node_type[0], degree0 = degree[0];
#pragma omp parallel for schedule(static) reduction(| : type_differs, type_all, degree_differs, degree_all) if (N > PACK_PARALLEL)
    for (int64_t i = 0; i < N; ++i) {
        type_differs |= node_type[i] ^ type0;
        type_all |= node_type[i];
        degree_differs |= degree[i] ^ degree0;
        degree_all |= degree[i];
    }
#pragma omp parallel for schedule(static) reduction(| : edge_all) if (E > PACK_PARALLEL)
    for (int64_t i = 0; i < 2 * E; ++i) edge_all |= edge[i];
#pragma omp parallel for schedule(static) reduction(max : largest) if (G > PACK_PARALLEL)
    for (int64_t g = 0; g < G; ++g) largest = n_nodes[g] > largest ? n_nodes[g] : largest;
    const int summed = largest <= PACK_SUMMED || (int64_t)largest * PACK_SUMMED_SHARE <= N;
    index_bad = !summed;
#pragma omp parallel for schedule(static) reduction(| : index_bad, empty) if (N > PACK_PARALLEL)
    for (int64_t g = 0; g < G; ++g) {
        const int64_t first = node_index[g], n = n_nodes[g];
        empty |= n == 0;
        /* the graphs' nodes have to follow one another from 0 to N (and lie inside the arrays, whatever the graphs before say) */
        if (first + n > N || first + n != (g + 1 < G ? (int64_t)node_index[g + 1] : N) || (g == 0 && first != 0)) {
            index_bad |= 1;
            continue;
        }
        if (!summed) continue;
        edge_start[g] = n > 0 ? edge_index[first] : 0;
        uint32_t expected = edge_start[g], bad = 0;
        for (int64_t i = 0; i < n; ++i) {
            bad |= edge_index[first + i] ^ expected;
            expected += degree[first + i];
        }
        index_bad |= bad != 0;
    }
    plan[PLAN_TYPE_BYTES] = bytes_for(type_differs, type_all);
    plan[PLAN_TYPE_VALUE] = type0;
    plan[PLAN_DEGREE_BYTES] = bytes_for(degree_differs, degree_all);
    plan[PLAN_DEGREE_VALUE] = degree0;
    plan[PLAN_INDEX_FOLLOWS] = index_bad == 0;
    plan[PLAN_EDGE_BYTES] = edge_all < 65536 ? 2 : 4;
    plan[PLAN_EMPTY_GRAPH] = empty;
}

/* Word w of a row's negated literals alone: bit b is the complement of positive bit 32 w + b - hv, 0 outside 0 .. hv - 1. */
static inline uint32_t negated_word(const uint32_t *p, int32_t words, uint32_t last, int32_t hv, int32_t w) {
    const int32_t from = w * 32 - hv;
    if (from <= -32) return 0;
    const int32_t low = from >= 0 ? from / 32 : -1, shift = from & 31;
    uint32_t out = low >= 0 && low < words ? (~p[low] & (low == words - 1 ? last : 0xFFFFFFFFu)) >> shift : 0;
    if (shift && low + 1 < words) out |= (~p[low + 1] & (low + 1 == words - 1 ? last : 0xFFFFFFFFu)) << (32 - shift);
    return out;
}

/* The (hv + 31) / 32 words of each row that hold its positive literals, bits past them cleared.  Returns 0 if every
 * row is what those words say it is (negated literals their complements, all other bits 0), else 1. */
int gtm_pack_rows(const uint32_t *X, int64_t rows, int32_t LA, int32_t hv, uint32_t *out) {
    uint32_t bad = 0;
    const int32_t words = (hv + 31) / 32;
    if (hv % 32 == 0) {
#pragma omp parallel for schedule(static) reduction(| : bad) if (rows * LA > PACK_PARALLEL)
        for (int64_t r = 0; r < rows; ++r) {
            const uint32_t *x = X + r * LA;
            uint32_t *o = out + r * words;
            for (int32_t w = 0; w < words; ++w) {
                o[w] = x[w];
                bad |= ~(x[w] ^ x[w + words]);
            }
        }
    } else {
        const uint32_t last = (1u << (hv % 32)) - 1u;
#pragma omp parallel for schedule(static) reduction(| : bad) if (rows * LA > PACK_PARALLEL)
        for (int64_t r = 0; r < rows; ++r) {
            const uint32_t *x = X + r * LA;
            uint32_t *o = out + r * words;
            for (int32_t w = 0; w < words; ++w) o[w] = w + 1 < words ? x[w] : x[w] & last;
            for (int32_t w = words - 1; w < LA; ++w)
                bad |= x[w] ^ ((w < words ? o[w] : 0u) | negated_word(o, words, last, hv, w));
        }
    }
    return bad != 0;
}

/* n numbers, `bytes` (1, 2 or 4) of each. */
void gtm_pack_numbers(const uint32_t *in, int64_t n, int32_t bytes, void *out) {
    if (bytes == 1) {
        uint8_t *o = out;
#pragma omp parallel for schedule(static) if (n > 4 * PACK_PARALLEL)
        for (int64_t i = 0; i < n; ++i) o[i] = (uint8_t)in[i];
    } else if (bytes == 2) {
        uint16_t *o = out;
#pragma omp parallel for schedule(static) if (n > 4 * PACK_PARALLEL)
        for (int64_t i = 0; i < n; ++i) o[i] = (uint16_t)in[i];
    } else {
        const int64_t piece = 1 << 16;
#pragma omp parallel for schedule(static) if (n > 4 * piece)
        for (int64_t a = 0; a < n; a += piece) memcpy((uint32_t *)out + a, in + a, (size_t)(n - a < piece ? n - a : piece) * 4);
    }
}

/* A new array's pages are made by whoever first writes to them; done by all threads while the device still works on what goes there. */
void gtm_touch_pages(void *array, int64_t bytes) {
#pragma omp parallel for schedule(static) if (bytes > 4 * PACK_PARALLEL)
    for (int64_t at = 0; at < bytes; at += 4096) ((volatile char *)array)[at] = 0;
}

#define OUTPUTS_4(v) { (v) & 1, ((v) >> 1) & 1, ((v) >> 2) & 1, ((v) >> 3) & 1 }
/* Clause outputs, which cross the bus as bits: out[i] = bit i % 32 of word i / 32.  Four outputs per table look-up; from
 * PACK_PARALLEL words on by all threads (a new array's pages are then also touched by all of them). */
void gtm_unpack_outputs(const uint32_t *bits, int64_t n, int32_t *out) {
    static const int32_t of_half_byte[16][4] = {OUTPUTS_4(0), OUTPUTS_4(1), OUTPUTS_4(2), OUTPUTS_4(3), OUTPUTS_4(4), OUTPUTS_4(5),
                                                OUTPUTS_4(6), OUTPUTS_4(7), OUTPUTS_4(8), OUTPUTS_4(9), OUTPUTS_4(10), OUTPUTS_4(11),
                                                OUTPUTS_4(12), OUTPUTS_4(13), OUTPUTS_4(14), OUTPUTS_4(15)};
    const int64_t piece = 1 << 10, words = n / 32;
#pragma omp parallel for schedule(static) if (words > PACK_PARALLEL / 4)
    for (int64_t a = 0; a < words; a += piece)
        for (int64_t w = a; w < words && w < a + piece; ++w)
            for (int q = 0; q < 8; ++q) memcpy(out + 32 * w + 4 * q, of_half_byte[(bits[w] >> (4 * q)) & 0xF], 16);
    for (int64_t i = 32 * words; i < n; ++i) out[i] = (bits[words] >> (i % 32)) & 1;
}
