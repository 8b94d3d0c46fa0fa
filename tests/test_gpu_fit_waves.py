"""Depth-1 training with a wave per clause, and with the clauses' lists of rows in LDS: at the edges of what each takes -
rows of 1 to 64 words, 16 and 17 literal words, 63 and 64 classes, clauses longer than their list - every split follows
the oracle bit for bit (whole numbers: no tolerance)."""

import numpy as np
import pytest

from oracle import gtm_oracle as o
from tests import helpers

pytestmark = pytest.mark.gpu


def follow(graphs, tune, switches, classes, clauses, kernel, state_bits=8, density=0.05, s=3.0, max_included=None):
    from tests.gpu_harness import Device, profiled

    for name, value in switches.items():
        tune(name, value)
    cfg = helpers.oracle_config(graphs, classes=classes, clauses=clauses, T=30, state_bits=state_bits, max_included=max_included)
    model = helpers.random_model(7, cfg, 1, s=s, include_density=density)
    # dense random clauses hold nowhere: a third of them get includes that one node satisfies
    rng = np.random.default_rng(3)
    for c in range(0, cfg.clauses, 3):
        if graphs.number_of_nodes:
            keep = graphs.X[int(rng.integers(graphs.number_of_nodes))].copy()
            model.ta_state[c, :, cfg.state_bits - 1] &= keep
    dev = Device(model, graphs)
    assert dev.build_tiles()
    G = graphs.number_of_graphs
    Y = o.encode_labels(rng.integers(0, classes, size=G), classes, cfg.threshold)
    for epoch in range(2):
        o.fit(model, graphs, Y)
        with profiled() as kernels:
            dev.fit(Y, 0, G, epoch * G)
        assert kernels() == {kernel: 1}
        ta, _, w = dev.download()
        assert np.array_equal(w, model.clause_weights), "weights after epoch %d" % epoch
        assert np.array_equal(ta, model.ta_state), "automata after epoch %d" % epoch


@pytest.mark.parametrize("sizes,hv_size,classes", [
    ([1, 31, 32, 0, 3], 20, 2),                # one word; literals that do not fill their last word
    ([512, 480, 33, 511, 1], 256, 10),         # 16 words a row, 16 literal words: the last shape of eight groups of lanes
    ([513, 1024, 40, 0, 700], 256, 3),         # 17 to 32 words: four groups
    ([1025, 2048, 64, 65, 1999], 32, 5),       # 33 to 64 words: two groups
    ([300, 257, 290, 12], 264, 10),            # 17 literal words: the automata in LDS
    ([90, 64, 33, 80], 64, 63),
    ([90, 64, 33, 80], 64, 64),
], ids=str)
@pytest.mark.parametrize("switches,state_bits,density", [
    ({}, 8, 0.05), ({}, 6, 0.6), ({}, 12, 0.3), ({"GTM_NO_FIT_WAVES": "1"}, 8, 0.3),
    ({"GTM_NO_FIT_WAVES": "1", "GTM_FIT_LIST_ROWS": "0"}, 8, 0.3), ({"GTM_NO_FIT_WAVES": "1", "GTM_FIT_LIST_ROWS": "64"}, 6, 0.3),
], ids=["waves", "waves-6-bits", "waves-12-bits", "lists-in-lds", "no-lists", "lists-too-short"])
def test_lists_of_rows_at_their_edges(sizes, hv_size, classes, switches, state_bits, density, tune):
    graphs = helpers.random_graphs(len(sizes) + hv_size, n_graphs=3 * len(sizes), sizes=sizes * 3, hv_size=hv_size, n_symbols=9, max_degree=0,
                                   node_types=("a", "b") if classes == 3 else ("a",))
    waves = hv_size <= 256 and classes <= 63 and "GTM_NO_FIT_WAVES" not in switches
    follow(graphs, tune, switches, classes, clauses=21, kernel=b"k_fit_waves" if waves else b"k_fit_persistent", state_bits=state_bits, density=density,
           max_included=20 if state_bits == 6 else None)


@pytest.mark.parametrize("hv_size,max_nodes", [(512, 1), (520, 2), (2048, 1)])
@pytest.mark.parametrize("s,per_group", [(1.0, None), (5.0, "20")])  # (of 128 words 15 fit in LDS)
def test_feedback_of_many_literal_words(hv_size, max_nodes, s, per_group, tune):
    """Single nodes and pairs of thousands of literals: Type I bits a byte per thread, feedback of the clauses that get any."""
    graphs = helpers.random_graphs(hv_size, n_graphs=30, max_nodes=max_nodes, hv_size=hv_size, n_symbols=40, max_degree=0)
    if per_group is not None and hv_size == 2048:
        per_group = "15"
    follow(graphs, tune, {} if per_group is None else {"GTM_FIT_PER_GROUP": per_group}, classes=10, clauses=45, kernel=b"k_fit_persistent",
           density=0.02, s=s)


@pytest.mark.parametrize("sizes,hv_size,clauses,kernel", [
    ([5, 3, 0, 1, 4], 4800, 20, b"k_fit_persistent"),    # 300 words: rows of as many literals have no room
    ([3, 5, 2], 3300, 2100, b"k_fit_persistent"),         # nine clauses a workgroup: nor have lists
    ([32, 31, 7, 0, 1], 512, 21, b"k_fit_persistent"),    # 32 words, 32 nodes: the last graphs tested node by node
    ([32, 31, 7, 0, 1], 496, 21, b"k_fit_persistent"),    # 31 words: the first on rows
    ([17, 16, 2], 264, 21, b"k_fit_persistent"),          # 17 words
    ([17, 16, 2], 256, 21, b"k_fit_waves"),
], ids=str)
@pytest.mark.parametrize("density", [0.003, 0.3])
def test_few_nodes_of_many_literals(sizes, hv_size, clauses, kernel, density, tune):
    """Graphs of a few nodes whose words are too many for a wave per clause: one launch, whatever the number of literals."""
    graphs = helpers.random_graphs(hv_size, n_graphs=3 * len(sizes), sizes=sizes * 3, hv_size=hv_size, n_symbols=30, max_degree=0,
                                   node_types=("a", "b", "c"))
    follow(graphs, tune, {}, classes=3, clauses=clauses, kernel=kernel, density=density)
