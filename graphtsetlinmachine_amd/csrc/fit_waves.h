// A whole run of training examples of a depth-1 model in one cooperative launch, one wave per clause.
//
// The scheme and the exchange are those of fit_persistent.h; here a workgroup owns at most 16 clauses, one per wave,
// and a clause's state lives in its wave's registers for the whole run: lane w holds the planes of automaton word w,
// lane k the weight of class k and its class's random words, and what the wave decides from - included literals, picked
// node, feedback of the classes - is the same for all lanes.  LDS holds the rows of this and the next graph, the
// clauses' lists of rows (fit_lists.h), and what crosses waves: votes, class sums, labels.
//
// A step is a chain of dependent instructions of a few waves, four to five clocks each, and every step waits for the
// slowest of all clauses, so what counts is the longest wave: random words are drawn while the class sums travel,
// the words of the picked node arrive meanwhile, a list is made anew from the include words in registers, and
// nothing that the step needs is divided, looked up twice or fetched from memory on that chain.
//
// 361 nodes, 2,500 clauses of 8 words on 250 workgroups, us per example in the first epochs of 3,000 and over 60,000 examples: 10.1 and 9.5
// with the clauses' state in LDS, their include planes walked on the scalar unit and the whole graph's literal words staged; 3.9 and
// 4.1 now (8 to 16 clauses per workgroup alike), of which about 2.5 are the exchange - an add and a look at memory that all XCDs
// share, and the slowest of 250 workgroups.  32 workgroups take 3.2.
#pragma once

constexpr int FITV_MAX_WORDS = 16;    // automaton words: four lanes draw the Type I bits of one
constexpr int FITV_MAX_CLASSES = 63;  // lane 63 draws for the node pick

inline size_t fit_waves_lds_words(int per_group, int rows_words, int lists) {
    return ((size_t)per_group * lists / 2 + 3) / 4 * 4 + 2 * (size_t)rows_words;
}

template <int MAXB, bool EXACT>
__global__ __launch_bounds__(FITP_BLOCK) void k_fit_waves(FitPersistParams p) {
    extern __shared__ __align__(16) uint32_t lds[];
    __shared__ int32_t votes[64], sums[64], labels[2][64];
    __shared__ int go_on;
    constexpr int WAVES = FITP_BLOCK / 64, POLL = WAVES - 1;  // the last wave adds the votes to the class sums and polls
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int LA = p.LA, B = EXACT ? MAXB : p.B, K = p.K;
    const int c = (int)blockIdx.x * p.clauses_per_group + wave;
    const bool owns = wave < p.clauses_per_group && c < p.C;  // (the same for the whole wave)
    const int last = p.first_example + p.n_examples - 1;
    const int all_rows = p.literals + p.n_types + 1, ones_row = all_rows - 1, type_row = p.literals + c % p.n_types;
    const unsigned long long everyone = (unsigned long long)gridDim.x;

    uint16_t *list = (uint16_t *)lds + (size_t)wave * p.lists;
    uint32_t *rows_both = lds + ((size_t)p.clauses_per_group * p.lists / 2 + 3) / 4 * 4;  // [2][p.rows_words]

    // the wave's clause -> registers
    uint32_t planes[MAXB] = {};
    int32_t weight = 0;
    if (owns) {
        if (lane < LA) {
#pragma unroll
            for (int b = 0; b < MAXB; ++b)
                if (EXACT || b < B) planes[b] = p.bank[((int64_t)c * LA + lane) * B + b];
        }
        if (lane < K) weight = p.weights[(int64_t)lane * p.C + c];
    }
    fits_word<MAXB, EXACT> word(planes, B);
    int entries = 0;  // of the list: the node-type row and the included literals
    auto make_list = [&]() {
        uint32_t mine = lane < LA ? word.top() : 0u;
        if (lane == LA - 1) mine &= p.filter;
        if (lane == 0) list[0] = (uint16_t)type_row;
        entries = fitl_append(mine, LA, 0, list, p.lists, 1, lane);
        fitl_finish(list, p.lists, entries, ones_row, p.lanes_log, lane);
        fitp_wave_lds_sync();
    };
    // lanes k < K: the gates of class k for this step; lane 63: the node pick of the next
    philox_out drawn = {};
    auto draw = [&](uint32_t step) {
        const bool pick = lane == 63;
        drawn = philox4x32_10((uint32_t)c, pick ? 0u : (uint32_t)lane, pick ? step + 1u : step,
                              pick ? (uint32_t)GTM_TAG_CLAUSE_NODE : (uint32_t)GTM_TAG_CLAUSE_UPDATES, p.k0, p.k1);
    };

    int n_now = (int)p.n_nodes[p.first_example], n_next = (int)p.n_nodes[min(p.first_example + 1, last)];
    uint32_t base_now = p.node_index[p.first_example], base_next = p.node_index[min(p.first_example + 1, last)];
    FitGraph fg = fit_graph_slot(p.tg, p.first_example, n_now);
    auto rows_of = [&](const FitGraph &f) { return p.tiles + (int64_t)f.tile * p.tg.rows * p.tg.tw + f.word0; };
    if (owns) {
        make_list();
        draw(p.first_step - 1u);  // (the pick of the first step)
    }
    {
        FitRowLoader all;
        all.prepare(fg.words, FITP_BLOCK, tid);
        all.request(rows_of(fg), p.tg.tw, all_rows, fg.words, rows_both + wave * 64, FITP_BLOCK, tid);
    }
    if (tid < 64) {
        votes[lane] = 0;
        if (lane < K) labels[0][lane] = p.encoded_Y[(int64_t)p.first_example * K + lane];
        if (lane == 0) go_on = 1;
    }
    __builtin_amdgcn_s_waitcnt(FITP_WAIT_VMEM);
    lds_barrier();

    // node count (even lanes) and first node (odd lanes) of a graph: a value per lane, so that nothing waits for it before it is used
    const uint32_t *sizes = lane & 1 ? p.node_index : p.n_nodes;
    constexpr int LOADERS = POLL * 64;  // threads that request the next graph's rows
    FitRowLoader loader{};
    int loader_words = 0;
    int quarter_log = 2;  // 2^quarter_log >= 4 LA lanes draw the Type I bits of one class
    while ((1 << quarter_log) < 4 * LA) ++quarter_log;
    const int place = 2 * (lane & ((1 << p.lanes_log) - 1));
    const int item = lane & ((1 << quarter_log) - 1), nth = lane >> quarter_log, at_once = 64 >> quarter_log;
    // polling lane k: class k's word as it stood when the slots of this step and the next two were last complete
    unsigned long long seen[3] = {};
    unsigned long long *slot_now = p.class_sum;
    int slot = 0;

    for (int i = 0; i < p.n_examples; ++i) {
        const uint32_t step = p.first_step + (uint32_t)i;
        // ---- 1. the wave's clause on the graph: truth (K1), node (K7), votes (K6)
        int node = -1;
        bool fired = false;
        if (owns) {
            const int stride = fitl_stride(fg.words);
            const uint32_t *col = rows_both + (i & 1) * p.rows_words + (place < stride ? place : 0);
            const uint2 v = fitl_nodes(fitl_truth(list, entries, col, stride, p.lanes_log, lane), fg, p.lanes_log, lane);
            if (n_now > 0) node = fitl_pick_node(v, (uint32_t)__builtin_amdgcn_readlane(drawn.v[0], 63), lane);
            fired = n_now == 0 || node >= 0;  // (the reference's arithmetic for a graph without nodes, kernels.py:289-295)
            if (fired && lane < K) atomicAdd(&votes[lane], weight);
        }
        lds_barrier();  // the group's votes are complete

        // ---- 2. class sums across the device (see fit_persistent.h); meanwhile all that does not need them
        if (wave == POLL && lane < K) {
            __hip_atomic_fetch_add(&slot_now[(lane * FITP_SUM_PARTS + (int)(blockIdx.x % FITP_SUM_PARTS)) * FITP_SUM_STRIDE],
                                   FITP_ARRIVED + (unsigned long long)(long long)votes[lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            votes[lane] = 0;
        }
        uint32_t x = 0u;  // the picked node's literal words, lane w word w
        if (owns && node >= 0 && lane < LA) x = p.X[((int64_t)base_now + node) * LA + lane];
        const int ex = p.first_example + i;
        const FitGraph fn = fit_graph_slot(p.tg, min(ex + 1, last), n_next);
        const uint32_t after = sizes[min(ex + 2, last)];
        if (wave != POLL && i + 1 < p.n_examples) {
            if (fn.words != loader_words) loader_words = fn.words, loader.prepare(fn.words, LOADERS, tid);
            loader.request(rows_of(fn), p.tg.tw, all_rows, fn.words, rows_both + (~i & 1) * p.rows_words + wave * 64, LOADERS, tid);
            if (wave == POLL - 1 && lane < K)
                fitp_load_to_lds((const uint32_t *)p.encoded_Y + (int64_t)(ex + 1) * K + lane, (uint32_t *)labels[~i & 1]);
        }
        if (owns) draw(step);
        if (wave == POLL && lane < K) {
            uint32_t polls = 0;
            unsigned long long waiting_since = 0ull, sum = 0ull;
            bool ok = !p.force_abort;
            if (!ok) __hip_atomic_store(p.abort_flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            while (ok) {
                // the abort flag travels with the parts: asked for after a look in vain it was a second round trip per look
                unsigned long long part[FITP_SUM_PARTS];
#pragma unroll
                for (int s = 0; s < FITP_SUM_PARTS; ++s)
                    part[s] = __hip_atomic_load(&slot_now[(lane * FITP_SUM_PARTS + s) * FITP_SUM_STRIDE], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
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
        __builtin_amdgcn_s_waitcnt(FITP_WAIT_VMEM);  // the next graph's words are in LDS
        lds_barrier();
        if (!go_on) break;  // uniform over the group; every group leaves at its next check

        // ---- 3. feedback (K8) and automaton updates (K9), all of it in the clause's wave
        if (owns) {
            int u = 0;
            if (lane < K) {
                int cs = sums[lane];
                const int y = labels[i & 1][lane];
                cs = cs > p.T ? p.T : (cs < -p.T ? -p.T : cs);
                const int target = 1 - 2 * (cs > y);
                const int sign = weight >= 0 ? 1 : -1;
                int err = y - cs;
                err = err < 0 ? -err : err;
                const bool skip = (target == -1 && (uint64_t)drawn.v[0] >= p.q_thr) ||
                                  ((uint64_t)drawn.v[1] * (uint64_t)(2 * (int64_t)p.T) >= ((uint64_t)err << 32));
                u = skip ? 0 : target * sign;
                if (u > 0 && node >= 0 && (weight < 0 ? -(int64_t)weight : (int64_t)weight) < 2147483647) {
                    weight += sign;
                } else if (u < 0 && node >= 0) {
                    weight -= sign;
                    if (p.negative == 0 && weight < 1) weight = 1;
                }
            }
            const unsigned long long type1 = __ballot(u > 0), type2 = __ballot(u < 0);
            if ((type1 | type2) != 0ull) {
                const uint32_t was = word.top();
                const bool hit = node >= 0, learns = hit && entries - 1 <= p.max_included;
                unsigned long long to_draw = type1;
                uint32_t bits = 0u;  // Type I bits of `ready` classes: word w of the j-th of them in lane (j << quarter_log) + 4 w
                int ready = 0, used = 0;
                for (unsigned long long m = type1 | type2; m != 0ull; m &= m - 1) {
                    uint32_t up = hit ? ~x & ~word.top() : 0u, down = 0u;
                    if (m & (0ull - m) & type1) {
                        if (used == ready) {
                            unsigned long long mine = to_draw;
                            for (int skip = 0; skip < nth; ++skip) mine &= mine - 1;
                            bits = 0u;
                            if (mine != 0ull)
                                bits = fitl_feedback_byte(p.k0, p.k1, (uint32_t)c, (uint32_t)item >> 2, (uint32_t)item & 3u, step, 0u,
                                                          (uint32_t)(__ffsll((long long)mine) - 1), p.thr16)
                                       << (8 * (item & 3));
                            bits |= (uint32_t)__builtin_amdgcn_mov_dpp((int)bits, 0xB1, 0xF, 0xF, true);  // lanes of a quad: [1, 0, 3, 2]
                            bits |= (uint32_t)__builtin_amdgcn_mov_dpp((int)bits, 0x4E, 0xF, 0xF, true);  // [2, 3, 0, 1]
                            for (ready = 0; ready < at_once && to_draw != 0ull; ++ready) to_draw &= to_draw - 1;
                            used = 0;
                        }
                        const uint32_t fb = (uint32_t)__builtin_amdgcn_ds_bpermute(4 * ((used << quarter_log) + 4 * lane), (int)bits);
                        ++used;
                        up = learns ? (p.boost == 1 ? x : x & ~fb) : 0u;
                        down = learns ? ~x & fb : fb;
                    }
                    word.count(up, down);
                }
                uint32_t changed = lane < LA ? word.top() ^ was : 0u;
                if (lane == LA - 1) changed &= p.filter;
                if (__ballot(changed != 0u) != 0ull) make_list();
            }
        }
        // (the wave goes straight on to the next graph: everything that its evaluation reads was complete at the barrier above)
        slot = slot == 2 ? 0 : slot + 1;
        slot_now = p.class_sum + (size_t)slot * K * FITP_SUM_PARTS * FITP_SUM_STRIDE;
        fg = fn;
        n_now = n_next, base_now = base_next;
        n_next = __builtin_amdgcn_readlane(after, 0), base_next = (uint32_t)__builtin_amdgcn_readlane(after, 1);
    }
    __builtin_amdgcn_s_waitcnt(FITP_WAIT_VMEM);  // no load into LDS is left in flight when the group ends
    lds_barrier();
    // own state -> global memory (also after an abort: every clause is left as of some whole step)
    if (owns) {
        if (lane < LA) word.store(p.bank + ((int64_t)c * LA + lane) * B);
        if (lane < K) p.weights[(int64_t)lane * p.C + c] = weight;
    }
}
