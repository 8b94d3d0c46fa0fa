"""The tiles of a data set, word for word: a model with one clause per (literal, node type) shows, through
``transform_nodewise`` on the tiles, every literal at every node."""

import numpy as np
import pytest

from tests import helpers

pytestmark = pytest.mark.gpu

SHAPES = [
    # one literal word, several graphs per word, graphs without nodes among them, three node types
    dict(seed=1, g=dict(hv_size=10, sizes=[3, 0, 1, 16, 7, 2, 0, 5], node_types=("a", "b", "c"))),
    # two words (loads of 4 bytes), tiles that end inside a group of 8 words, more than one tile
    dict(seed=2, g=dict(hv_size=32, n_graphs=700, max_nodes=12)),
    # literals that are no multiple of 32, with a quad of literal words that is only partly there
    dict(seed=3, g=dict(hv_size=50, sizes=[33, 0, 64, 1, 31, 32, 65, 40])),
    dict(seed=4, g=dict(hv_size=200, n_symbols=20, sizes=[70, 17, 40, 96])),
    # half tiles: 4 and 8 words per node (one or both quads hold positive literals)
    dict(seed=5, g=dict(hv_size=64, n_graphs=40, max_nodes=90, min_nodes=20), half=True),
    dict(seed=6, g=dict(hv_size=128, n_graphs=23, max_nodes=361, min_nodes=300, max_degree=0), half=True),
    # one node per graph and thousands of literals: one tile whose literals are shared out among workgroups ...
    dict(seed=7, g=dict(hv_size=600, n_symbols=30, n_graphs=37, max_nodes=1)),
    # ... and more literal words than one workgroup counts in its LDS
    dict(seed=8, g=dict(hv_size=4500, n_symbols=30, n_graphs=5, max_nodes=2)),
]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "build%d" % s["seed"])
def test_every_literal_of_every_node_is_in_the_tiles(shape):
    from graphtsetlinmachine_amd.tm import MultiClassGraphTsetlinMachine

    g = dict(shape["g"])
    g.setdefault("n_graphs", len(g.get("sizes", ())))
    graphs = helpers.random_graphs(shape["seed"], **g)
    literals, types = 2 * graphs.hypervector_size, graphs.number_of_node_types()
    clauses, chunks, top = literals * types, (literals - 1) // 32 + 1, 7
    bank = np.zeros((clauses, chunks, 8), dtype=np.uint32)
    literal = np.arange(clauses) // types  # clause c looks at nodes of type c % types
    bank[np.arange(clauses), literal // 32, top] = np.uint32(1) << (literal % 32).astype(np.uint32)
    tm = MultiClassGraphTsetlinMachine(clauses, 100, 1.0, seed=1)
    tm.set_state((bank, np.ones((1, clauses), dtype=np.int32), 1, clauses, literals, 1, 8, chunks, None, None))
    got, sums = tm.transform_nodewise(graphs)
    bits = (graphs.X[:, np.arange(literals) // 32] >> (np.arange(literals) % 32).astype(np.uint32)) & 1
    for g in range(graphs.number_of_graphs):
        a = int(graphs.node_index[g])
        n = int(graphs.number_of_graph_nodes[g])
        want = bits[a:a + n][:, literal].T * (graphs.node_type[a:a + n][None, :] == (np.arange(clauses) % types)[:, None])
        assert np.array_equal(got[g, :, :n], want), g
        assert not got[g, :, n:].any()
        assert sums[g, 0] == (clauses if n == 0 else (want.sum(axis=1) > 0).sum())
    dg = tm._test_graphs
    assert dg.tiles is not None
    if not shape.get("half"):
        # the last words of the buffer: the literals, rarest first (a graph without nodes holds every literal once)
        count = bits.sum(axis=0, dtype=np.int64) + int((graphs.number_of_graph_nodes == 0).sum())
        assert np.array_equal(dg.tiles.cpu().numpy()[-literals:], np.lexsort((np.arange(literals), count)))
