"""Message rows made by shifting rows (data sets whose edges are a few moves): class sums and clause outputs equal
the oracle's, and the kernel is the one taken - or not, where the edges are too many kinds of moves."""

import ctypes

import numpy as np
import pytest

from oracle import gtm_oracle as o
from tests import helpers

pytestmark = pytest.mark.gpu


def _graphs(sizes, moves, seed, hv=20):
    """Nodes n of every graph get an edge to n + d of type t for each (t, d) in `moves` that stays in the graph
    (about one in eight is left out)."""
    from graphtsetlinmachine_amd.graphs import Graphs

    rng = np.random.default_rng(seed)
    np.random.seed(seed)
    g = Graphs(len(sizes), symbols=list(range(9)), hypervector_size=hv, hypervector_bits=2)
    g.number_of_graph_nodes[:] = sizes
    g.prepare_node_configuration()
    node_of = np.concatenate([np.arange(n) for n in sizes]).astype(np.int64)
    size_of = np.repeat(sizes, sizes)
    graph_of = np.repeat(np.arange(len(sizes)), sizes)
    there = [(node_of + d >= 0) & (node_of + d < size_of) & (rng.random(node_of.size) < 0.875) for _, d in moves]
    g.add_graph_nodes(sum(m.astype(np.uint32) for m in there))
    g.prepare_edge_configuration()
    for (t, d), m in zip(moves, there):
        g.add_graph_node_edges(graph_of[m], node_of[m], node_of[m] + d, "type%d" % t)
    for _ in range(2):
        nodes = np.flatnonzero(rng.random(node_of.size) < 0.7)
        g.add_graph_node_properties(nodes, rng.integers(0, 9, size=nodes.size))
    g.encode()
    return g


GRID = [(0, -29), (1, 29), (2, -1), (3, 1)]
SHAPES = [
    ("pairs", [2] * 700, [(0, 1), (0, -1)], dict(message_size=256), True),
    ("tiny_with_loops", [1, 16, 0, 7, 2] * 40, [(0, 0), (1, 3), (0, -2)], dict(message_size=37), True),
    ("ragged_chains", [3, 41, 17, 0, 33, 32, 64, 1] * 30, [(0, -1), (1, 1)], dict(message_size=128), True),
    ("odd_messages", [70, 31, 65, 96, 0], [(0, -1), (1, 1)], dict(message_size=45), True),
    ("long_chains", [1000, 999, 513], [(0, -1), (1, 1)], dict(message_size=512), True),
    ("grid", [841] * 5, GRID, dict(message_size=1024), True),
    ("far_moves", [300, 257, 290], [(0, 32), (1, -64), (2, 96), (3, -33), (0, 255), (1, -250), (2, 63), (3, 0)],
     dict(message_size=64), True),
    ("types_beyond_the_messages", [50, 64, 20], [(t, (-1) ** t * t) for t in range(6)], dict(message_size=4), True),
    ("too_many", [50, 64, 20], [(0, d) for d in range(-4, 5)], dict(message_size=64), False),
]


@pytest.mark.parametrize("complementary", [False, True], ids=["", "complementary"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: s[0])
def test_rows_by_moves(shape, complementary):
    from bench import read_kernel_breakdown, read_kernel_profile
    from graphtsetlinmachine_amd import _abi
    from graphtsetlinmachine_amd.tm import _ptr, _stream
    from tests.gpu_harness import Device

    import torch

    name, sizes, moves, sizing, taken = shape
    graphs = _graphs(np.array(sizes), moves, seed=len(name))
    cfg = helpers.oracle_config(graphs, classes=3, clauses=70, depth=3, T=50, message_bits=2, **sizing)
    model = helpers.random_model(7, cfg, 3, include_density=0.03, message_density=0.3 / sizing["message_size"])
    dev = Device(model, graphs)
    if complementary and not dev.declare_complementary():
        pytest.skip("graphs without nodes: never declared complementary")
    assert dev.build_tiles()
    n = graphs.number_of_graphs
    want = o.score(model, graphs)
    nbytes = _abi.lib.gtm_moves_bytes(ctypes.byref(dev.acfg), ctypes.byref(dev.dg.desc))
    buffer = torch.full((nbytes // 4,), 0x5A5A5A5A, dtype=torch.int32, device="cuda")
    _abi.call("gtm_build_moves", ctypes.byref(dev.acfg), ctypes.byref(dev.dg.desc), _ptr(buffer), _stream())
    _abi.call("gtm_profile_enable", 1)
    try:
        got = dev.score(0, n, n)
        torch.cuda.synchronize()
        kernels = [k for k, _, _ in read_kernel_breakdown()]
        read_kernel_profile()
    finally:
        _abi.call("gtm_profile_enable", 0)
    assert np.array_equal(got, want)
    assert ("k_tile_messages_moved" in kernels) == taken
    assert np.array_equal(dev.score(0, n, 2), want)  # launch groups: tiles from the middle of the data set


def test_scoring_captured_on_another_stream():
    """Class sums of a data set that was brought to the device on the default stream, captured in a graph on the capture's own
    stream and replayed, with eager work in between."""
    from graphtsetlinmachine_amd.tm import MultiClassGraphTsetlinMachine

    import torch

    name, sizes, moves, sizing, _ = SHAPES[5]
    graphs = _graphs(np.array(sizes * 3), moves, seed=3)  # (enough edges for the moves to be looked for)
    tm = MultiClassGraphTsetlinMachine(60, 50, 2.0, depth=3, seed=5, **sizing)
    tm.fit(graphs, np.arange(len(sizes) * 3) % 3, epochs=1)
    want = tm.score_device(graphs).cpu().numpy()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = tm.score_device(graphs)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy(), want)
        assert np.array_equal(tm.score_device(graphs).cpu().numpy(), want)


def test_moves_are_looked_for_by_the_first_call_that_uses_them():
    """Training has no use for them; scoring the training set has, and so has every layout of its tiles."""
    from graphtsetlinmachine_amd.tm import MultiClassGraphTsetlinMachine

    name, sizes, moves, sizing, _ = SHAPES[5]
    graphs = _graphs(np.array(sizes * 3), moves, seed=3)
    tm = MultiClassGraphTsetlinMachine(60, 50, 2.0, depth=3, seed=5, **sizing)
    tm.fit(graphs, np.arange(len(sizes) * 3) % 3, epochs=1)
    dg = tm._train_graphs
    assert dg.tiles is not None and dg.moves is None
    want = tm.score(graphs)
    assert tm._train_graphs is dg and dg.moves is not None
    dg._tiles_key = None
    tm.fit(graphs, np.arange(len(sizes) * 3) % 3, epochs=0, incremental=True)
    assert dg.moves is None
    features, sums = tm.transform(graphs)
    assert dg.moves is not None and np.array_equal(sums, want)
    words = dg.moves[:9].cpu().numpy()  # the (type, offset) keys found, then whether there were too many
    assert sorted(int(v) for v in words[:4]) == sorted((t << 16) | (32768 + d) for t, d in GRID) and not words[4:].any()


def test_without_room_for_the_moves_the_edges_are_walked(monkeypatch):
    import torch

    from graphtsetlinmachine_amd.tm import MultiClassGraphTsetlinMachine

    name, sizes, moves, sizing, _ = SHAPES[5]
    graphs = _graphs(np.array(sizes * 3), moves, seed=3)
    tm = MultiClassGraphTsetlinMachine(60, 50, 2.0, depth=3, seed=5, **sizing)
    tm.fit(graphs, np.arange(len(sizes) * 3) % 3, epochs=1)
    want, dg, empty = tm.score(graphs), tm._train_graphs, torch.empty
    assert dg.moves is not None
    words = dg.moves.numel()
    dg._tiles_key = None

    def refuse(*size, **kwargs):
        if size == (words,):
            raise torch.OutOfMemoryError("no room")
        return empty(*size, **kwargs)

    monkeypatch.setattr(torch, "empty", refuse)
    assert np.array_equal(tm.score(graphs), want) and dg.moves is None
    assert np.array_equal(tm.score(graphs), want)
