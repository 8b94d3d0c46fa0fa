"""The one-workgroup training kernel: every way of spreading a step over its lanes gives the oracle's trajectory."""

import numpy as np
import pytest

from oracle import gtm_oracle as o
from tests import helpers

pytestmark = pytest.mark.gpu

# lanes per (clause, node): 16 and 1 (one pair, many pairs); node pick and decisions by one wave and by several;
# messages straight along the edges and through the nodes' vectors (many edges); include planes copied (8 bits) and, where
# the copy does not fit beside the automata (262 clauses of 2 bits), in place; random draws of one example at a time (5,500
# decisions); words that no power of two divides
SHAPES = [
    dict(seed=1, clauses=1, classes=1, depth=2, message_size=256, g=dict(n_graphs=20, max_nodes=1, max_degree=2)),
    dict(seed=2, clauses=10, classes=2, depth=2, message_size=256, g=dict(n_graphs=40, max_nodes=2, hv_size=32)),
    dict(seed=3, clauses=13, classes=5, depth=3, message_size=96, g=dict(sizes=[5, 0, 3, 1, 0, 8] * 4, hv_size=50, edge_types=("a", "b"))),
    dict(seed=4, clauses=33, classes=2, depth=2, message_size=32, g=dict(n_graphs=10, max_nodes=64, min_nodes=60, max_degree=9)),
    dict(seed=5, clauses=70, classes=3, depth=2, message_size=64, max_included=4, g=dict(n_graphs=12, max_nodes=20, node_types=("p", "q", "r"))),
    dict(seed=6, clauses=40, classes=2, depth=2, message_size=160, state_bits=11, g=dict(n_graphs=16, max_nodes=7)),
    dict(seed=8, clauses=275, classes=20, depth=2, message_size=32, g=dict(n_graphs=6, max_nodes=4, hv_size=16)),
    dict(seed=7, clauses=262, classes=2, depth=3, message_size=320, state_bits=2, g=dict(n_graphs=8, max_nodes=6)),
]


@pytest.mark.parametrize("s", [1.0, 3.0])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "spread%d" % s["seed"])
def test_every_spread_trains_as_the_oracle(shape, s):
    from tests.gpu_harness import Device

    g = dict(shape["g"])
    g.setdefault("n_graphs", len(g.get("sizes", ())))
    graphs = helpers.random_graphs(shape["seed"], **g)
    depth = shape["depth"]
    cfg = helpers.oracle_config(graphs, classes=shape["classes"], clauses=shape["clauses"], depth=depth, T=15,
                                message_size=shape["message_size"], state_bits=shape.get("state_bits", 8),
                                max_included=shape.get("max_included"))
    model = helpers.random_model(shape["seed"], cfg, depth, s=(s,) * depth, include_density=0.03)
    dev = Device(model, graphs)
    G = graphs.number_of_graphs
    Y = o.encode_labels(np.random.default_rng(shape["seed"]).integers(0, shape["classes"], size=G), shape["classes"], cfg.threshold)
    for epoch in range(3):
        o.fit(model, graphs, Y)
        dev.fit(Y, 0, G, epoch * G)
        ta, banks, w = dev.download()
        assert np.array_equal(w, model.clause_weights), "weights after epoch %d" % epoch
        assert np.array_equal(ta, model.ta_state), "layer-0 automata after epoch %d" % epoch
        for layer in range(depth - 1):
            assert np.array_equal(banks[layer], model.message_ta_state[layer]), "bank %d epoch %d" % (layer, epoch)


def _trains_as_the_oracle(model, dev, graphs, classes, seed, epochs=2):
    G = graphs.number_of_graphs
    Y = o.encode_labels(np.random.default_rng(seed).integers(0, classes, size=G), classes, model.cfg.threshold)
    for epoch in range(epochs):
        o.fit(model, graphs, Y)
        dev.fit(Y, 0, G, epoch * G)
        ta, banks, w = dev.download()
        assert np.array_equal(w, model.clause_weights), "weights after epoch %d" % epoch
        assert np.array_equal(ta, model.ta_state), "layer-0 automata after epoch %d" % epoch
        for layer in range(model.depth - 1):
            assert np.array_equal(banks[layer], model.message_ta_state[layer]), "bank %d epoch %d" % (layer, epoch)


@pytest.mark.parametrize("degree", [2, 9], ids=["few", "many"])
@pytest.mark.parametrize("order", ["reversed", "shuffled", "gap"])
def test_edges_that_do_not_lie_node_after_node(order, degree):
    """The same graphs with a node's edges anywhere in the edge array: edge_index says where."""
    import copy

    from tests.gpu_harness import Device

    graphs = helpers.random_graphs(11, n_graphs=30, max_nodes=20, max_degree=degree, edge_types=("a", "b"))
    cfg = helpers.oracle_config(graphs, classes=2, clauses=8, depth=2, T=15, message_size=64)
    model = helpers.random_model(11, cfg, 2, s=2.0, include_density=0.03)
    moved = copy.deepcopy(graphs)
    N, gap = len(graphs.node_type), 5 if order == "gap" else 0
    nodes = np.arange(N)[::-1] if order == "reversed" else np.random.default_rng(3).permutation(N) if order == "shuffled" else np.arange(N)
    edges, at = [], 0
    for n in nodes:
        a, k = int(graphs.edge_index[n]), int(graphs.number_of_graph_node_edges[n])
        moved.edge_index[n] = at
        edges.append(graphs.edge[a:a + k])
        edges.append(np.zeros((gap, 2), dtype=np.uint32))
        at += k + gap
    moved.edge = np.ascontiguousarray(np.concatenate(edges))
    _trains_as_the_oracle(model, Device(model, moved), graphs, 2, 11)
