"""Class sums of small models on graphs of a few nodes in one launch (k_score_small): at the edges of what it takes the sums
equal the oracle's and those of the general path, and what it does not take is scored as before (whole numbers: no tolerance)."""

import ctypes

import numpy as np
import pytest

from oracle import gtm_oracle as o
from tests import helpers

pytestmark = pytest.mark.gpu

SHAPES = [
    # nodes per graph, hypervector size, node types, edge types, most edges of a node, model, taken
    ([2], 32, 1, 1, 1, dict(classes=2, clauses=10, depth=2, message_size=256, message_bits=2), True),
    ([1, 0, 2, 1], 16, 2, 3, 2, dict(classes=8, clauses=7, depth=3, message_size=32, message_bits=1), True),
    ([8, 1, 0, 7, 5], 128, 3, 40, 5, dict(classes=32, clauses=65, depth=2, message_size=32, message_bits=3), True),
    ([5, 3], 65, 5, 70, 9, dict(classes=3, clauses=40, depth=4, message_size=160, message_bits=2), True),
    ([3, 0], 50, 11, 2, 0, dict(classes=1, clauses=33, depth=3, message_size=128, message_bits=2), True),  # no edges at all
    ([1], 64, 1, 1, 0, dict(classes=64, clauses=20, depth=1), True),        # 16 slots a graph for its classes
    ([7, 8], 100, 2, 1, 0, dict(classes=11, clauses=9, depth=1), True),
    ([9, 1], 32, 1, 1, 1, dict(classes=2, clauses=10, depth=2, message_size=256), False),   # a node too many
    ([2], 129, 1, 1, 1, dict(classes=2, clauses=10, depth=2, message_size=256), False),     # a literal word too many
    ([2], 32, 1, 1, 1, dict(classes=2, clauses=10, depth=2, message_size=288), False),      # a message word too many
    ([2], 32, 1, 1, 1, dict(classes=2, clauses=10, depth=2, message_size=37), False),
    ([2], 32, 1, 1, 1, dict(classes=65, clauses=10, depth=2, message_size=64), False),
    ([2], 128, 1, 1, 1, dict(classes=2, clauses=400, depth=3, message_size=256), False),    # LDS
]


@pytest.mark.parametrize("sizes,hv,node_types,edge_types,degree,sizing,taken", SHAPES, ids=lambda v: str(v) if isinstance(v, list) else "")
@pytest.mark.parametrize("n_graphs,state_bits", [(1, 8), (67, 6), (403, 8)])
def test_class_sums_in_one_launch(sizes, hv, node_types, edge_types, degree, sizing, taken, n_graphs, state_bits, tune):
    from graphtsetlinmachine_amd import _abi
    from tests.gpu_harness import Device

    nodes = (sizes * n_graphs)[:n_graphs]
    if max(nodes) != max(sizes):
        nodes[0] = max(sizes)
    graphs = helpers.random_graphs(hv, n_graphs=n_graphs, sizes=nodes, hv_size=hv, n_symbols=9, max_degree=degree,
                                   node_types=["t%d" % i for i in range(node_types)], edge_types=["e%d" % i for i in range(edge_types)])
    cfg = helpers.oracle_config(graphs, state_bits=state_bits, T=30, **{k: v for k, v in sizing.items() if k != "depth"})
    model = helpers.random_model(5, cfg, sizing["depth"], include_density=0.02, message_density=0.01)
    for bank in [model.ta_state] + model.message_ta_state:  # two thirds of the clauses with at most one literal a bank: they hold somewhere
        bank[::3, :, state_bits - 1] = 0
        bank[1::3, 1:, state_bits - 1] = 0
        bank[1::3, 0, state_bits - 1] &= np.uint32(1 << 5)
    dev = Device(model, graphs)
    assert bool(_abi.lib.gtm_score_needs_tiles(ctypes.byref(dev.acfg), ctypes.byref(dev.dg.desc))) != taken
    want = o.score(model, graphs)
    kernel, launches, total = ctypes.c_char_p(), ctypes.c_int32(), ctypes.c_double()
    _abi.call("gtm_profile_enable", 1)
    got = dev.score(0, n_graphs, n_graphs)
    _abi.call("gtm_profile_read", ctypes.byref(kernel), ctypes.byref(launches), ctypes.byref(total))
    _abi.call("gtm_profile_enable", 0)
    assert (kernel.value == b"k_score_small") == taken, kernel.value
    assert np.array_equal(got, want)
    first = n_graphs // 3
    assert np.array_equal(dev.score(first, n_graphs - first, 5), want[first:])
    assert (want != 0).any()
    tune("GTM_NO_SMALL_SCORE", "1")
    assert np.array_equal(dev.score(0, n_graphs, n_graphs), want)


@pytest.mark.parametrize("nodes,hv,classes,depth,clauses,most", [
    (2, 32, 2, 2, 100, 32 * (1250000 // (100 * 5))),                # pairs: 32 to a workgroup, a quad of literals and four of a layer
    (1, 32, 2, 2, 100, 64 * (2500000 // (100 * 6))),                # single nodes count their second class in a turn of its own
    (8, 128, 2, 3, 10, 8 * 1300),                                   # graphs of eight: workgroups ...
    (8, 128, 2, 3, 200, 8 * (750000 // (200 * 10))),                # ... and quads
    (4, 16, 2, 1, 200, 16 * 640), (1, 128, 1, 1, 100, 64 * 640),    # depth 1: workgroups
    (4, 16, 2, 1, 201, 0), (1, 128, 1, 1, 101, 0),                  # ... and quads of clauses
])
def test_large_data_sets_stay_on_tiles(nodes, hv, classes, depth, clauses, most):
    from graphtsetlinmachine_amd import _abi

    cfg = _abi.make_config(classes=classes, clauses=clauses, literals=2 * hv, state_bits=8, boost_true_positive_feedback=1, threshold=10, q=1.0,
                           max_included_literals=64, negative_clauses=1, max_nodes=nodes, message_size=256, message_bits=2, depth=depth,
                           s=(1.0,) * depth, seed=1)
    d = _abi.GraphsDesc()
    d.number_of_node_types, d.max_number_of_graph_nodes = 1, nodes
    d.number_of_graphs = most
    assert most == 0 or not _abi.lib.gtm_score_needs_tiles(ctypes.byref(cfg), ctypes.byref(d))
    d.number_of_graphs += 1
    assert _abi.lib.gtm_score_needs_tiles(ctypes.byref(cfg), ctypes.byref(d))
