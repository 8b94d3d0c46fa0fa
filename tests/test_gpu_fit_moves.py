"""Training with message layers on data sets whose edges are a few moves (k_fit_moves): automata of every bank and the
weights follow the oracle bit for bit in every layout, and other data sets keep the kernel that walks the edges."""

import ctypes

import numpy as np
import pytest

from oracle import gtm_oracle as o
from tests import helpers
from tests.test_gpu_message_moves import GRID, _graphs

pytestmark = pytest.mark.gpu

CHAIN = [(0, -1), (1, 1)]
SHAPES = [
    # name, nodes per graph, moves, hypervector size, model, taken
    ("tiny_with_loops", [1, 16, 0, 7, 2] * 4, [(0, 0), (1, 3), (0, -2)], 20, dict(classes=2, clauses=33, depth=2, message_size=32, message_bits=3), True),
    ("chains_of_one_word", [31, 17, 32, 0, 24, 20] * 2, CHAIN, 40, dict(classes=64, clauses=40, depth=3, message_size=96), True),
    ("ragged_chains", [3, 41, 17, 33, 32, 64, 1, 200], CHAIN, 20, dict(classes=3, clauses=300, depth=4, message_size=64, message_bits=1), True),
    ("long_chains", [1000, 999, 513, 1], CHAIN, 64, dict(classes=2, clauses=200, depth=2, message_size=512), True),
    ("longest_rows", [2048, 1025, 2000], CHAIN, 16, dict(classes=2, clauses=60, depth=2, message_size=256), True),
    ("grid", [841] * 3, GRID, 128, dict(classes=10, clauses=70, depth=3, message_size=288), True),
    ("grid_of_many_clauses", [841] * 2, GRID, 40, dict(classes=4, clauses=1500, depth=2, message_size=64), True),
    ("far_moves", [300, 257, 290], [(0, 32), (1, -64), (2, 96), (3, -33), (0, 255), (1, -250), (2, 63), (3, 0)], 33,
     dict(classes=3, clauses=50, depth=3, message_size=64), True),
    ("no_edges", [70, 31, 65, 0], [], 20, dict(classes=3, clauses=20, depth=3, message_size=32), False),
    ("too_many", [90, 84, 70], [(0, d) for d in range(-4, 5)], 20, dict(classes=3, clauses=40, depth=2, message_size=64), False),
]
LAYOUTS = {
    "as_it_comes": {},
    "in_memory": {"GTM_FIT_DEEP_IN_MEMORY": "1"},
    "7_a_workgroup_dealt_every_3_examples": {"GTM_FIT_DEEP_CLAUSES_PER_GROUP": "7", "GTM_FIT_DEEP_CHUNK": "3"},
    "40_a_workgroup_in_memory": {"GTM_FIT_DEEP_CLAUSES_PER_GROUP": "40", "GTM_FIT_DEEP_IN_MEMORY": "1"},
    "17_a_workgroup": {"GTM_FIT_DEEP_CLAUSES_PER_GROUP": "17"},
}


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: s[0])
@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("boost,max_included,state_bits", [(1, None, 8), (0, 9, 5), (1, None, 12)])
def test_training_by_moves(shape, layout, boost, max_included, state_bits, tune):
    import torch

    from tests.gpu_harness import Device, profiled

    name, sizes, moves, hv, sizing, taken = shape
    for switch, value in LAYOUTS[layout].items():
        tune(switch, value)
    tune("GTM_NO_SMALL_FIT", "1")
    graphs = _graphs(np.array(sizes), moves, seed=len(name), hv=hv)
    depth = sizing["depth"]
    cfg = helpers.oracle_config(graphs, T=30, boost=boost, max_included=max_included, state_bits=state_bits, **sizing)
    model = helpers.random_model(5, cfg, depth, s=(3.0, 2.0, 1.5, 1.2)[:depth], include_density=0.02, message_density=0.02)
    dev = Device(model, graphs)
    assert dev.build_tiles()
    G = graphs.number_of_graphs
    Y = o.encode_labels(np.random.default_rng(1).integers(0, cfg.classes, size=G), cfg.classes, cfg.threshold)
    for epoch in range(2):
        o.fit(model, graphs, Y)
        with profiled() as kernels:
            dev.fit(Y, 0, G // 3, epoch * G)  # the restart from memory is covered, too
            dev.fit(Y, G // 3, G - G // 3, epoch * G + G // 3)
        assert all(k.startswith(b"k_fit_moves<") == taken for k in kernels()), kernels()
        if taken and "17" not in layout and layout != "as_it_comes":
            assert all((b"in memory" in k) == ("memory" in layout or cfg.classes > 63) for k in kernels()), kernels()
        own = max(-(-cfg.clauses // torch.cuda.get_device_properties(0).multi_processor_count), int(LAYOUTS[layout].get("GTM_FIT_DEEP_CLAUSES_PER_GROUP", 1)))
        collected = 4 * own * len(moves) * cfg.message_bits > cfg.message_size
        assert all((b"sent rows in LDS" in k) == (b"in memory" in k and collected) for k in kernels() if taken), kernels()
        ta, banks, w = dev.download()
        assert np.array_equal(w, model.clause_weights), "weights after epoch %d" % epoch
        assert np.array_equal(ta, model.ta_state), "layer-0 automata after epoch %d" % epoch
        for layer in range(depth - 1):
            assert np.array_equal(banks[layer], model.message_ta_state[layer]), "bank %d epoch %d" % (layer, epoch)


# The shares of a workgroup's 16 waves and 128 lanes' words that a clause in registers can have: clauses per workgroup, automaton words per clause
# (literals / 32 + 2 message banks), hence waves per clause, a lane's words, and whether the rows of two graphs fit in LDS beside the lists.
REGISTER_SHAPES = [
    ("two_waves_two_words_rows_in_place", 324, 1024, 1024, 8, b"k_fit_moves<registers, rows in place>"),   # 192 words, 128 lanes
    ("four_waves_one_word_rows_in_place", 324, 1024, 1024, 4, b"k_fit_moves<registers, rows in place>"),   # 192 words, 256 lanes
    ("two_waves_two_words_staged_rows", 90, 448, 448, 8, b"k_fit_moves<registers>"),                     
    ("one_wave_one_word", 90, 256, 256, 16, b"k_fit_moves<registers>"),                                   # 48 words, 64 lanes; the polling wave owns a clause
    ("one_wave_two_words", 90, 384, 384, 16, b"k_fit_moves<registers>"),                                  # 72 words
    ("one_wave_all_128_words", 70, 512, 768, 9, b"k_fit_moves<registers>"),                               # 32 + 2 * 48
    ("one_wave_129_words", 70, 520, 768, 9, b"k_fit_moves<in memory>"),                                   # 33 + 2 * 48: too many
]


@pytest.mark.parametrize("name,nodes,hv,message_size,per_group,kernel", REGISTER_SHAPES, ids=lambda v: v if isinstance(v, str) else "")
@pytest.mark.parametrize("state_bits", [8, 6])
def test_clauses_in_registers_at_every_share_of_the_waves(name, nodes, hv, message_size, per_group, kernel, state_bits, tune):
    from tests.gpu_harness import Device, profiled

    tune("GTM_FIT_DEEP_CLAUSES_PER_GROUP", str(per_group))
    tune("GTM_NO_SMALL_FIT", "1")
    moves = GRID if nodes == 324 else CHAIN
    graphs = _graphs(np.array([nodes, nodes, nodes if nodes == 324 else 33, nodes]), moves, seed=nodes + hv, hv=hv)
    cfg = helpers.oracle_config(graphs, classes=5, clauses=2 * per_group + 3, depth=3, message_size=message_size, T=30, state_bits=state_bits)
    model = helpers.random_model(5, cfg, 3, s=(3.0, 2.0, 1.5), include_density=0.004, message_density=0.004)
    dev = Device(model, graphs)
    assert dev.build_tiles()
    Y = o.encode_labels(np.arange(4) % 5, 5, cfg.threshold)
    for epoch in range(2):
        o.fit(model, graphs, Y)
        with profiled() as kernels:
            dev.fit(Y, 0, 4, epoch * 4)
        assert list(kernels()) == [kernel], kernels()
        ta, banks, w = dev.download()
        assert np.array_equal(w, model.clause_weights) and np.array_equal(ta, model.ta_state)
        assert all(np.array_equal(a, b) for a, b in zip(banks, model.message_ta_state))


@pytest.mark.parametrize("in_memory", [False, True])
@pytest.mark.parametrize("switches,kernels_expected", [
    ({"GTM_NO_FIT_MOVES": "1"}, {"k_fit_deep_persistent": 4}),
    # launches that start three examples into a kernel's run or later give up: each trains on three, the next goes on from there
    ({"GTM_FIT_SPIN_LIMIT": "from 3"}, {"k_fit_moves": 2, "k_fit_deep_persistent": 2}),
    ({"GTM_FIT_SPIN_LIMIT": "from 9"}, {"k_fit_moves": 4, "k_fit_deep_persistent": 1}),
    ({"GTM_FIT_SPIN_LIMIT": "from 0"}, {"k_fit_moves": 1, "k_fit_deep_persistent": 1}),
], ids=["edges-walked", "both-give-up", "moves-give-up-at-the-end", "both-give-up-at-once"])
def test_another_kernel_goes_on_where_one_gave_up(switches, kernels_expected, in_memory, tune):
    """Chains train on k_fit_moves; where it is off or gives up, on the kernel that walks the edges, and where that gives up, on
    launches per example: the same automata and weights, each example once."""
    from tests.gpu_harness import Device, profiled

    for name, value in switches.items():
        tune(name, value)
    if in_memory:
        tune("GTM_FIT_DEEP_IN_MEMORY", "1")
    tune("GTM_FIT_DEEP_CLAUSES_PER_GROUP", "7")  # (clauses are dealt out anew every three examples)
    tune("GTM_FIT_DEEP_CHUNK", "3")
    graphs = _graphs(np.array([100, 90, 110, 70, 65, 33, 100, 128, 80, 1, 77]), CHAIN, seed=2)
    cfg = helpers.oracle_config(graphs, classes=3, clauses=40, depth=3, message_size=64, T=30)
    model = helpers.random_model(5, cfg, 3, s=(3.0, 2.0, 1.5), include_density=0.02, message_density=0.02)
    dev = Device(model, graphs)
    assert dev.build_tiles()
    Y = o.encode_labels(np.arange(11) % 3, 3, cfg.threshold)
    for epoch in range(2):
        o.fit(model, graphs, Y)
        with profiled() as kernels:
            dev.fit(Y, 0, 11, epoch * 11)
        ran = {}
        for k, launches in kernels().items():
            one_launch = [n for n in ("k_fit_moves", "k_fit_deep_persistent") if k.startswith(n.encode())]
            if one_launch:
                assert (b"in memory" in k) == in_memory
                ran[one_launch[0]] = launches
        assert ran == kernels_expected, kernels()
        ta, banks, w = dev.download()
        assert np.array_equal(w, model.clause_weights), "weights after epoch %d" % epoch
        assert np.array_equal(ta, model.ta_state), "automata after epoch %d" % epoch
        assert all(np.array_equal(a, b) for a, b in zip(banks, model.message_ta_state))


@pytest.mark.parametrize("in_memory", [False, True])
def test_giving_up_leaves_the_model_as_it_was(in_memory, tune):
    from graphtsetlinmachine_amd import _abi
    from tests.gpu_harness import Device

    if in_memory:
        tune("GTM_FIT_DEEP_IN_MEMORY", "1")
    graphs = _graphs(np.array([100, 90, 110]), CHAIN, seed=2)
    cfg = helpers.oracle_config(graphs, classes=3, clauses=40, depth=3, message_size=64, T=30)
    model = helpers.random_model(5, cfg, 3, s=(3.0, 2.0, 1.5), include_density=0.02, message_density=0.02)
    dev = Device(model, graphs)
    assert dev.build_tiles()
    Y = o.encode_labels(np.arange(3) % 3, 3, cfg.threshold)
    tune("GTM_FIT_SPIN_LIMIT", "abort")
    with pytest.raises(_abi.GtmError, match="gave up waiting.*as it was before the call"):
        dev.fit(Y, 0, 3, 0)
    tune("GTM_FIT_SPIN_LIMIT", None)
    for trained in (False, True):
        if trained:
            o.fit(model, graphs, Y)
            dev.fit(Y, 0, 3, 0)
        ta, banks, w = dev.download()
        assert np.array_equal(w, model.clause_weights) and np.array_equal(ta, model.ta_state)
        assert all(np.array_equal(a, b) for a, b in zip(banks, model.message_ta_state))


def test_more_rows_than_a_list_can_number():
    """65,600 node types and as many clauses: the type rows of the last of them have numbers of 17 bits, lists hold 16."""
    from oracle import gtm_oracle_c as oc
    from tests.gpu_harness import Device

    graphs = _graphs(np.array([7, 4, 9, 1, 16]), CHAIN, seed=4, hv=32)
    types = 65600
    graphs.node_type_id = {"type %d" % t: t for t in range(types)}
    graphs.node_type[:] = np.random.default_rng(2).choice([0, 3, 65471, 65472, 65500, 65535, 65536, 65599], size=graphs.node_type.size)
    cfg = helpers.oracle_config(graphs, classes=2, clauses=types, message_size=32, T=30000)
    model = helpers.random_model(5, cfg, 2, s=(3.0, 2.0), include_density=0.0, message_density=0.0)
    dev = Device(model, graphs)
    assert dev.build_tiles()
    Y = o.encode_labels(np.arange(5) % 2, 2, cfg.threshold)
    for epoch in range(2):
        oc.fit(model, graphs, Y)
        dev.fit(Y, 0, 5, epoch * 5)
        ta, banks, w = dev.download()
        assert np.array_equal(w, model.clause_weights) and np.array_equal(ta, model.ta_state)
        assert np.array_equal(banks[0], model.message_ta_state[0])


@pytest.mark.parametrize("in_memory", [False, True])
def test_without_room_for_masks_and_lists_the_edges_are_walked(in_memory, tune, monkeypatch):
    """What only k_fit_moves uses is asked for where it can run - not for data sets without edges, lists not where they stay in LDS - and
    a caller that has no more than the rest trains all the same."""
    import torch

    from graphtsetlinmachine_amd import _abi, tm as tm_module
    from tests.gpu_harness import Device

    clauses = 41
    if in_memory:
        tune("GTM_FIT_DEEP_CLAUSES_PER_GROUP", "20")
    graphs = _graphs(np.array([100, 90, 110, 64]), CHAIN, seed=2)
    size = lambda name, dev: getattr(_abi.lib, name)(ctypes.byref(dev.acfg), ctypes.byref(dev.dg.desc))
    extra = lambda dev: size("gtm_fit_workspace_bytes", dev) - size("gtm_fit_workspace_least_bytes", dev)
    cfg = helpers.oracle_config(graphs, classes=3, clauses=clauses, depth=3, message_size=64, T=30)
    make = lambda g: Device(helpers.random_model(5, cfg, 3, s=(3.0, 2.0, 1.5), include_density=0.02, message_density=0.02), g)
    dev = make(graphs)
    masks = 4 * 8 * 4 * 4  # examples, moves, words of the longest rows, bytes
    lists = 60 * (48 + 2 * 128) * 2 if in_memory else 0  # clauses of whole workgroups, entries of their three lists, bytes
    assert masks + lists <= extra(dev) < masks + lists + 512
    tune("GTM_NO_FIT_MOVES", "1")
    assert extra(dev) == 0
    tune("GTM_NO_FIT_MOVES", None)
    assert extra(make(_graphs(np.array([100, 90]), [], seed=2))) == 0

    assert dev.build_tiles()
    least, st = size("gtm_fit_workspace_least_bytes", dev), dev.state()
    Y = o.encode_labels(np.arange(4) % 3, 3, cfg.threshold)
    y = tm_module._to_device(np.ascontiguousarray(Y, dtype=np.int32))
    ws = torch.empty(least, dtype=torch.uint8, device="cuda")
    fit = lambda nbytes: _abi.call("gtm_fit", ctypes.byref(dev.acfg), ctypes.byref(dev.dg.desc), ctypes.byref(st), tm_module._ptr(y), 0, 4, 0,
                                   tm_module._ptr(ws), nbytes, tm_module._stream())
    with pytest.raises(_abi.GtmError, match="workspace of"):
        fit(least - 1)
    _abi.call("gtm_profile_enable", 1)
    fit(least)
    kernel, launches, total = ctypes.c_char_p(), ctypes.c_int32(), ctypes.c_double()
    _abi.call("gtm_profile_read", ctypes.byref(kernel), ctypes.byref(launches), ctypes.byref(total))
    _abi.call("gtm_profile_enable", 0)
    assert kernel.value.startswith(b"k_fit_deep_persistent"), kernel.value
    o.fit(dev.model, graphs, Y)
    ta, banks, w = dev.download()
    assert np.array_equal(w, dev.model.clause_weights) and np.array_equal(ta, dev.model.ta_state)
    assert all(np.array_equal(a, b) for a, b in zip(banks, dev.model.message_ta_state))

    asked = []

    def no_room(self, nbytes):
        asked.append(nbytes)
        if len(asked) == 1:
            raise torch.OutOfMemoryError("no room")
        return torch.empty(max(int(nbytes), 256), dtype=torch.uint8, device="cuda")

    monkeypatch.setattr(tm_module.CommonTsetlinMachine, "_workspace_of", no_room)
    states = []
    for attempt in range(2):  # (the second has room at once)
        asked[:] = [0] * attempt
        np.random.seed(3)
        tm = tm_module.MultiClassGraphTsetlinMachine(clauses, 30, 2.0, depth=3, message_size=64, message_bits=2, seed=3)
        tm.fit(graphs, np.array([0, 1, 2, 0]), epochs=2)
        states.append(tm.get_state())
        assert attempt == 1 or asked[1] < asked[0]
    assert np.array_equal(states[0][0], states[1][0]) and np.array_equal(states[0][1], states[1][1])
