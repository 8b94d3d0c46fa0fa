"""Performance cases: what programs have this package do, through ``fit``, ``score`` and ``transform``.

A case is one call (for ``serve`` two) on one model:

``score``      class sums of a data set that stays resident, as after every epoch of a training program
``serve``      class sums of batches that were not scored before: two batches in turn, each of which is
               brought to the device again because a model keeps one test set resident
``transform``, ``transform_nodewise``
               clause outputs as features, per graph and per node
``fit``        one epoch over a resident data set, going on from the state at hand

on one of five kinds of graphs, those of the package's own workloads with their sizes as parameters:

``pairs``      two nodes that exchange one message each way, label = XOR of their symbols
``images``     one node per binary image, a symbol per pixel
``patches``    a node per patch of a binary image: pixel symbols and thermometer-coded position, no edges
``chains``     token sequences with 'Left' and 'Right' edges, label = length of the one run of token 0
``grid``       a node per patch of a colour image, thermometer-coded channels, an edge to each neighbour

Models are trained before they are measured: how many literals clauses include, and at how many nodes they
hold, decides how much the kernels have to do.
"""

import numpy as np
from numpy.lib.stride_tricks import sliding_window_view

from graphtsetlinmachine_amd.graphs import Graphs
from graphtsetlinmachine_amd.tm import MultiClassGraphTsetlinMachine

# ------------------------------------------------------------------------- cases


def _case(op, kind, graphs, **sizes):
    case = dict(op=op, kind=kind, graphs=graphs, hv=128, hv_bits=2, clauses=2500, T=3125, s=10.0, depth=1,
                message_size=256, message_bits=2, classes=10, state_bits=8, max_included=0, trained=2000, epochs=1)
    case.update(sizes)
    return case


def _pairs(**sizes):
    return dict(hv=32, clauses=10, T=100, s=1.0, depth=2, classes=2, **sizes)


def _grid(**sizes):
    return dict(side=32, patch=4, levels=8, hv=1024, clauses=8000, T=10000, s=15.0, depth=3, message_size=1024, **sizes)


def listed():
    cases = [
        # A request of a few small graphs, new ones each time: launches, copies and host work are all there is.
        ("serve_few_pairs", _case("serve", "pairs", 16, **_pairs(trained=1000))),
        # The test pass of the smallest workload, a model of ten clauses with a message layer.
        ("score_pairs", _case("score", "pairs", 10000, **_pairs(trained=2000))),
        # The test pass on single-node graphs with thousands of literals: one clause per image, no nodes to share.
        ("score_images", _case("score", "images", 10000, side=28, hv=2048, trained=5000)),
        # The test pass of the convolutional workload, the benchmark's headline.
        ("score_patches", _case("score", "patches", 10000, side=28, patch=10, trained=5000)),
        # New images in batches, as a service gets them: upload and layout count as much as the clauses; odd sizes.
        ("serve_patches", _case("serve", "patches", 999, side=28, patch=9, clauses=1999, T=2500, trained=2000)),
        # The test pass on long chains: one message layer on graphs of a thousand nodes.
        ("score_chains", _case("score", "chains", 3000, shortest=1000, longest=1000, symbols=26, hv=64, clauses=200, T=400,
                               s=1.0, depth=2, message_size=512, classes=2, trained=500)),
        # The test pass of the largest model: 8,000 clauses, two message layers, 841 nodes of 2,048 literals.
        ("score_grid", _case("score", "grid", 1000, **_grid(trained=256, epochs=10))),
        # Clause outputs of ragged short sequences, three layers deep, as features for something else.
        ("transform_ragged_chains", _case("transform", "chains", 4001, shortest=3, longest=41, symbols=11, hv=96,
                                          clauses=333, T=600, s=3.0, depth=3, classes=3, trained=2000)),
        # Training epochs: each example waits for the one before it, so its latency is what counts.
        ("fit_pairs", _case("fit", "pairs", 5000, **_pairs())),
        ("fit_patches", _case("fit", "patches", 3000, side=28, patch=10)),
        ("fit_chains", _case("fit", "chains", 1000, shortest=1000, longest=1000, symbols=26, hv=64, clauses=200, T=400,
                             s=1.0, depth=2, message_size=512, classes=2)),
        ("fit_grid", _case("fit", "grid", 512, **_grid())),
    ]
    return [dict(case, name=name) for name, case in cases]


def _spread(rng, low, high):
    """A whole number between low and high, spread over its logarithm."""
    return int(round(low * (high / low) ** rng.random()))


def draw(rng):
    op = rng.choice(["score", "score", "serve", "transform", "transform_nodewise", "fit", "fit"])
    kind = rng.choice(["pairs", "images", "patches", "chains", "grid"])
    state_bits = rng.choice([8, 8, 8, 6, 10])
    if kind == "pairs":
        sizes = dict(hv=rng.choice([16, 32, 50, 128]), clauses=_spread(rng, 10, 200), s=rng.choice([1.0, 2.0]), depth=rng.choice([2, 2, 3]),
                     message_size=rng.choice([32, 64, 256]), classes=2, most=10000, example_us=20.0)
    elif kind == "images":
        sizes = dict(side=rng.randint(12, 28), hv=rng.choice([512, 1000, 2048]), clauses=_spread(rng, 100, 2500), s=rng.choice([5.0, 10.0]), most=10000,
                     example_us=20.0)
    elif kind == "patches":
        side = rng.randint(16, 28)
        sizes = dict(side=side, patch=rng.randint(5, min(12, side - 4)), hv=rng.choice([64, 128, 128, 200, 256]), clauses=_spread(rng, 200, 2500),
                     s=rng.choice([5.0, 10.0]), most=6000, example_us=25.0)
    elif kind == "chains":
        longest = _spread(rng, 10, 1200)
        sizes = dict(shortest=rng.choice([longest, max(4, longest // 3), 4]), longest=longest, symbols=rng.choice([5, 11, 26]), hv=rng.choice([32, 64, 96, 256]),
                     clauses=_spread(rng, 40, 400), s=rng.choice([1.0, 3.0]), depth=rng.choice([1, 2, 2, 3]),
                     message_size=rng.choice([64, 128, 256, 512]), classes=rng.choice([2, 3]), max_included=rng.choice([0, 0, 16]), most=4000, example_us=60.0)
    else:
        side = rng.randint(10, 24)
        sizes = dict(side=side, patch=rng.randint(2, 4), levels=rng.choice([3, 5, 8]), hv=rng.choice([256, 512, 1024]), clauses=_spread(rng, 200, 4000),
                     s=rng.choice([5.0, 15.0]), depth=rng.choice([1, 2, 3]), message_size=rng.choice([256, 512, 1024]), most=800, example_us=130.0)
    most, example_us = sizes.pop("most"), sizes.pop("example_us")
    if op == "fit":
        most = min(most, int(6e4 / example_us))
    graphs = _spread(rng, 8, most)
    if op == "transform":
        graphs = min(graphs, max(1, int(2e7) // sizes["clauses"]))
    if op == "transform_nodewise":
        graphs = min(graphs, max(1, int(2e7) // (sizes["clauses"] * _most_nodes(dict(sizes, kind=kind)))))
    sizes.setdefault("T", int(sizes["clauses"] * 1.25) + 5)
    trained = {"pairs": 1000, "images": 1000, "patches": 1000, "chains": 300, "grid": 200}[kind]
    return _case(op, kind, graphs, state_bits=state_bits, trained=trained, **sizes)


# ------------------------------------------------------------------------ graphs


def _most_nodes(case):
    kind = case["kind"]
    if kind in ("pairs", "images"):
        return kind == "pairs" and 2 or 1
    if kind == "chains":
        return case["longest"]
    return (case["side"] - case["patch"] + 1) ** 2


def _new(case, n, symbols, parent, seed):
    if parent is not None:
        return Graphs(n, init_with=parent)
    saved = np.random.get_state()
    np.random.seed(seed % (1 << 32))
    g = Graphs(n, symbols=symbols, hypervector_size=case["hv"], hypervector_bits=case["hv_bits"])
    np.random.set_state(saved)
    return g


def _no_edges(g, nodes):
    g.number_of_graph_nodes[:] = nodes
    g.prepare_node_configuration()
    g.add_graph_nodes(0)
    g.prepare_edge_configuration()


def _positions(dim):
    """Thermometer-coded row and column of every patch: [dim * dim][2 * dim], column and row symbols in turn."""
    at = np.arange(dim)
    reached = at[None, :] <= at[:, None]
    out = np.zeros((dim, dim, 2 * dim), dtype=np.uint8)
    out[:, :, 0::2] = reached[:, None, :]
    out[:, :, 1::2] = reached[None, :, :]
    return out.reshape(dim * dim, 2 * dim)


def _add_patches(g, pixels, patch, dim):
    """A node per patch of pixels [n][side][side][values]: its position and the values in it."""
    n, where = pixels.shape[0], _positions(dim)
    block = max(1, (1 << 26) // (dim * dim * (2 * dim + patch * patch * pixels.shape[3])))
    for a in range(0, n, block):
        part = pixels[a:a + block]
        windows = sliding_window_view(part, (patch, patch), axis=(1, 2)).reshape(part.shape[0], dim * dim, -1)
        member = np.concatenate([np.broadcast_to(where, (part.shape[0],) + where.shape), windows], axis=2)
        g.add_graph_node_property_matrix(a * dim * dim, member.reshape(-1, member.shape[2]))


def _build(case, n, rng, truth, parent, seed):
    """n graphs and their labels; `truth` is what the classes look like, drawn once for all of a model's data."""
    kind, classes = case["kind"], case["classes"]
    y = rng.integers(0, classes, size=n).astype(np.uint32)
    if kind == "pairs":
        g = _new(case, n, ["A", "B"], parent, seed)
        g.number_of_graph_nodes[:] = 2
        g.prepare_node_configuration()
        g.add_graph_nodes(1)
        g.prepare_edge_configuration()
        each = np.repeat(np.arange(n), 2)
        g.add_graph_node_edges(each, np.tile([0, 1], n), np.tile([1, 0], n), "Plain")
        first = rng.integers(0, 2, size=n)
        g.add_graph_node_properties(np.arange(2 * n), np.stack([first, first ^ y], axis=1).reshape(-1))
        y = np.where(rng.random(n) < 0.01, 1 - y, y).astype(np.uint32)
    elif kind == "images":
        side = case["side"]
        g = _new(case, n, list(range(side * side)), parent, seed)
        _no_edges(g, 1)
        pixels = (rng.random((n, side * side), dtype=np.float32) < truth.reshape(classes, -1)[y]) ^ (rng.random((n, side * side), dtype=np.float32) < 0.05)
        g.add_graph_node_property_matrix(0, pixels)
    elif kind == "patches":
        side, patch = case["side"], case["patch"]
        dim = side - patch + 1
        g = _new(case, n, list(range(2 * dim + patch * patch)), parent, seed)
        _no_edges(g, dim * dim)
        pixels = (rng.random((n, side, side), dtype=np.float32) < truth[y]) ^ (rng.random((n, side, side), dtype=np.float32) < 0.05)
        _add_patches(g, pixels[..., None].view(np.uint8), patch, dim)
    elif kind == "chains":
        g = _new(case, n, list(range(case["symbols"])), parent, seed)
        length = rng.integers(case["shortest"], case["longest"] + 1, size=n)
        g.number_of_graph_nodes[:] = length
        g.prepare_node_configuration()
        each = np.repeat(np.arange(n), length)
        start = np.cumsum(length) - length
        at = np.arange(each.size) - start[each]
        left, right = at > 0, at < length[each] - 1
        g.add_graph_nodes(left.astype(np.uint32) + right)
        g.prepare_edge_configuration()
        g.add_graph_node_edges(each[left], at[left], at[left] - 1, "Left")
        g.add_graph_node_edges(each[right], at[right], at[right] + 1, "Right")
        token = rng.integers(1, case["symbols"], size=each.size)
        begin = start + rng.integers(0, length - y)  # a run of y + 1 tokens 0 somewhere
        for k in range(classes):
            token[begin[y >= k] + k] = 0
        g.add_graph_node_properties(np.arange(each.size), token)
    else:
        side, patch, levels = case["side"], case["patch"], case["levels"]
        dim = side - patch + 1
        g = _new(case, n, list(range(2 * dim + patch * patch * 3 * levels)), parent, seed)
        g.number_of_graph_nodes[:] = dim * dim
        g.prepare_node_configuration()
        row, column = (v.reshape(-1) for v in np.mgrid[0:dim, 0:dim])
        ways = [("Up", row > 0, -dim), ("Down", row < dim - 1, dim), ("Left", column > 0, -1), ("Right", column < dim - 1, 1)]
        g.add_graph_nodes(np.tile(sum(there.astype(np.uint32) for _, there, _ in ways), n))
        g.prepare_edge_configuration()
        for way, there, step in ways:
            source = np.flatnonzero(there)
            g.add_graph_node_edges(np.repeat(np.arange(n), source.size), np.tile(source, n), np.tile(source + step, n), way)
        colour = truth[y] + 0.1 * rng.standard_normal((n, side, side, 3), dtype=np.float32)
        coded = colour[..., None] > ((np.arange(levels) + 1.0) / (levels + 1.0)).astype(np.float32)
        _add_patches(g, coded.reshape(n, side, side, 3 * levels).view(np.uint8), patch, dim)
    g.encode()
    return g, y


def _truth(case, rng):
    if case["kind"] in ("images", "patches"):
        return np.where(rng.random((case["classes"], case["side"], case["side"])) < 0.5, 0.8, 0.1).astype(np.float32)
    if case["kind"] != "grid":
        return None
    side = case["side"]
    yy, xx = np.mgrid[0:side, 0:side]
    out = np.zeros((case["classes"], side, side, 3))
    for one in out:
        for channel in range(3):
            for _ in range(3):
                cx, cy = rng.uniform(side / 8, side * 7 / 8, size=2)
                width = rng.uniform(side / 13, side / 5.3)
                one[:, :, channel] += rng.uniform(0.4, 1.0) * np.exp(-((xx - cx) ** 2 + (yy - cy) ** 2) / (2 * width * width))
    return np.clip(out, 0.0, 1.0).astype(np.float32)


# ------------------------------------------------------------------------ passes


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    truth = _truth(case, rng)
    saved = np.random.get_state()
    np.random.seed((seed + 1) % (1 << 32))
    tm = MultiClassGraphTsetlinMachine(
        case["clauses"], case["T"], case["s"], depth=case["depth"], message_size=case["message_size"], message_bits=case["message_bits"],
        number_of_state_bits=case["state_bits"], max_included_literals=case["max_included"] or None, seed=seed + 2)
    np.random.set_state(saved)
    fitting = case["op"] == "fit"
    g, y = _build(case, case["graphs"] if fitting else case["trained"], rng, truth, None, seed)
    y[0] = case["classes"] - 1  # the first fit counts the classes
    tm.fit(g, y, epochs=case["epochs"], incremental=True)
    if fitting:
        return dict(op="fit", tm=tm, graphs=g, labels=y)
    batches = [_build(case, case["graphs"], rng, truth, g, seed)[0] for _ in range(2 if case["op"] == "serve" else 1)]
    return dict(op=case["op"], tm=tm, batches=batches)


def run(state):
    tm = state["tm"]
    if state["op"] == "fit":
        tm.fit(state["graphs"], state["labels"], epochs=1, incremental=True)
        return dict(automata=tm.ta_state_gpu, messages=list(tm.message_ta_state_gpu), weights=tm.clause_weights_gpu)
    if state["op"] == "transform":
        return tm.transform(state["batches"][0])
    if state["op"] == "transform_nodewise":
        return tm.transform_nodewise(state["batches"][0])
    return [tm.score(batch) for batch in state["batches"]]


def work(case):
    """Bytes: the graphs once (literal words, node types, edges), the model once (its include bits; for fit all of
    its automata, read and written), the outputs once.  The operations are on bits: none of them is a flop."""
    graphs, nodes, classes = case["graphs"], _most_nodes(case), case["classes"]
    if case["kind"] == "chains":
        nodes = (case["shortest"] + case["longest"]) / 2
    words = (2 * case["hv"] + 31) // 32
    message_words = (case["depth"] - 1) * ((2 * case["message_size"] + 31) // 32)
    degree = {"pairs": 1, "images": 0, "patches": 0, "chains": 2, "grid": 4}[case["kind"]] if case["depth"] > 1 else 0
    data = graphs * (nodes * (4 * words + 4 + 8 * degree) + 4)
    bank = 4 * case["clauses"] * (words + message_words)
    weights = 4 * case["clauses"] * classes
    if case["op"] == "fit":
        return {"bytes": data + 4 * graphs + 2 * bank * case["state_bits"] + 2 * weights, "flops": 0}
    out = 4 * graphs * classes
    if case["op"] == "transform":
        out += 4 * graphs * case["clauses"]
    if case["op"] == "transform_nodewise":
        out += 4 * graphs * case["clauses"] * _most_nodes(case)
    batches = 2 if case["op"] == "serve" else 1
    return {"bytes": batches * (data + out) + bank + weights, "flops": 0}


def tolerance(case):
    """Every result is a whole number: sums of votes, clause outputs, automata."""
    return "exact"
