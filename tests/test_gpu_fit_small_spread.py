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


# out-degrees of every graph's nodes: edges shared out evenly among the threads whichever node they start from - one node with all of
# them, at either end or in the middle, nodes without any between them, as many as are parked and one more, one node only
DEGREES = [
    dict(degrees=[40] + [0] * 63, clauses=10, bits=2),
    dict(degrees=[0] * 30 + [17, 0, 0, 3] + [0] * 6, clauses=4, bits=4),
    dict(degrees=[0] * 63 + [256], clauses=1, bits=4),
    dict(degrees=[0] * 63 + [257], clauses=1, bits=2),
    dict(degrees=[64, 64, 64, 64], clauses=2, bits=2),
    dict(degrees=[1, 0] * 16, clauses=16, bits=4),
    dict(degrees=[6], clauses=33, bits=1),
    dict(degrees=[1] * 32 + [0] + [1] * 31, clauses=3, bits=3),
]


@pytest.mark.parametrize("shape", DEGREES, ids=lambda s: "%dx%d" % (len(s["degrees"]), sum(s["degrees"])))
def test_edges_of_a_few_nodes_or_of_all(shape):
    from graphtsetlinmachine_amd.graphs import Graphs
    from tests.gpu_harness import Device

    G, degrees, rng = 12, np.array(shape["degrees"]), np.random.default_rng(len(shape["degrees"]))
    N = len(degrees)
    np.random.seed(N)
    g = Graphs(G, symbols=list(range(5)), hypervector_size=16, hypervector_bits=2)
    g.number_of_graph_nodes[:] = N
    g.prepare_node_configuration()
    g.add_graph_nodes(np.tile(degrees, G).astype(np.uint32))
    g.prepare_edge_configuration()
    source = np.tile(np.repeat(np.arange(N), degrees), G)
    graph, to, kind = np.repeat(np.arange(G), degrees.sum()), rng.integers(0, N, size=source.size), rng.integers(0, 3, size=source.size)
    for t in range(3):
        m = kind == t
        g.add_graph_node_edges(graph[m], source[m], to[m], "type%d" % t)
    for _ in range(2):
        nodes = np.flatnonzero(rng.random(G * N) < 0.7)
        g.add_graph_node_properties(nodes, rng.integers(0, 5, size=nodes.size))
    g.encode()
    cfg = helpers.oracle_config(g, classes=2, clauses=shape["clauses"], depth=3, T=15, message_size=96, message_bits=shape["bits"])
    model = helpers.random_model(N, cfg, 3, s=2.0, include_density=0.01)
    _trains_as_the_oracle(model, Device(model, g), g, 2, N)


@pytest.mark.parametrize("hv, nodes", [(256, 64), (272, 64), (520, 31), (1000, 64)], ids=["1024", "1088", "1023", "4032"])
def test_graphs_of_more_literal_words_than_are_fetched_ahead(hv, nodes):
    """At most 1,024 literal words of the next graph wait in registers; ragged sizes in turn, so that a graph with more follows
    one with fewer and the other way round."""
    from tests.gpu_harness import Device

    graphs = helpers.random_graphs(hv, sizes=[nodes, 3, nodes, nodes - 1, 0, nodes, nodes], n_graphs=7, hv_size=hv, max_degree=2)
    cfg = helpers.oracle_config(graphs, classes=2, clauses=3, depth=2, T=15, message_size=64)
    model = helpers.random_model(hv, cfg, 2, s=2.0, include_density=0.005)
    _trains_as_the_oracle(model, Device(model, graphs), graphs, 2, hv)


# message words per half and lanes that share a pair: 4 and 1, 16 and 4, 64 and 16 (each lane's words come in fours: the form that
# takes a half at a time), 4 and 2, 12 and 2, 3 and 1, 2 and 8 (the general form); every number of state bits has its own kernels
@pytest.mark.parametrize("state_bits", [6, 8, 12, 20])
@pytest.mark.parametrize("message_size, clauses, nodes", [
    (128, 40, 12), (512, 12, 5), (2048, 1, 3), (128, 20, 5), (384, 12, 10), (96, 30, 14), (64, 5, 5),
], ids=lambda v: str(v))
def test_message_words_a_half_at_a_time_and_one_by_one(message_size, clauses, nodes, state_bits):
    from tests.gpu_harness import Device

    graphs = helpers.random_graphs(message_size, n_graphs=10, max_nodes=nodes, min_nodes=max(1, nodes - 2), hv_size=16, edge_types=("a", "b"))
    cfg = helpers.oracle_config(graphs, classes=2, clauses=clauses, depth=3, T=15, message_size=message_size, state_bits=state_bits)
    model = helpers.random_model(message_size + clauses, cfg, 3, s=2.0, include_density=0.02, message_density=0.5 / message_size)
    _trains_as_the_oracle(model, Device(model, graphs), graphs, 2, clauses)
