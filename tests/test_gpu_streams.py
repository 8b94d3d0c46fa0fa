"""One model called on several streams, without a device-wide wait between the calls."""

import numpy as np
import pytest

from tests.test_gpu_message_moves import GRID, _graphs

pytestmark = pytest.mark.gpu


def _model_and_sets():
    from graphtsetlinmachine_amd.tm import MultiClassGraphTsetlinMachine

    sets = [_graphs(np.array([841] * n), GRID, seed=n) for n in (40, 60, 50)]
    tm = MultiClassGraphTsetlinMachine(120, 100, 2.0, depth=3, message_size=256, seed=5)
    tm.fit(sets[0], np.arange(40) % 3, epochs=1)
    want = [tm.score(s) for s in sets]
    return tm, sets, want


def test_data_sets_scored_in_turn_on_two_streams():
    import torch

    tm, sets, want = _model_and_sets()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    # the training set stays resident; the other two replace one another: brought to the device on one stream, scored on
    # it and on the other, and given up while that pass may be running, with the memory wanted again at once
    got = []
    for turn in range(12):
        here, there = streams[turn % 2], streams[1 - turn % 2]
        which = 1 + turn % 2
        with torch.cuda.stream(here):
            got.append((which, tm.score_device(sets[which])))
        with torch.cuda.stream(there):
            got.append((which, tm.score_device(sets[which])))
            got.append((0, tm.score_device(sets[0])))
        with torch.cuda.stream(here):
            other = 3 - which
            got.append((other, tm.score_device(sets[other])))
            torch.full((1 << 20,), 0x5A5A5A5A, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    for which, sums in got:
        assert np.array_equal(sums.cpu().numpy().reshape(want[which].shape), want[which]), which


def test_trained_on_one_stream_from_an_upload_on_another():
    import torch

    tm, sets, _ = _model_and_sets()
    twin, _, _ = _model_and_sets()
    y = np.arange(60) % 3
    tm.fit(sets[1], y, epochs=2, incremental=True)
    want = tm.score(sets[2])
    with torch.cuda.stream(torch.cuda.Stream()):
        twin.score_device(sets[1])
        sums = twin.score_device(sets[2])
    with torch.cuda.stream(torch.cuda.Stream()):
        twin.fit(sets[1], y, epochs=2, incremental=True)
        assert np.array_equal(twin.get_weights(), tm.get_weights())
    assert np.array_equal(twin.get_state()[0], tm.get_state()[0])
    assert np.array_equal(twin.score(sets[2]), want)
    del sums


def test_a_data_set_that_is_not_on_the_device_is_refused_under_capture():
    """... with an error, and the model goes on; so is one without this model's tiles, and one whose upload is under way."""
    import torch

    from graphtsetlinmachine_amd import _abi

    tm, sets, want = _model_and_sets()
    new = _graphs(np.array([841] * 30), GRID, seed=30)
    resident = tm._test_graphs
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        here = torch.zeros(1, device="cuda")
        with pytest.raises(_abi.GtmError, match="not on the device yet"):
            tm.score_device(new)
    assert tm._test_graphs is resident and here is not None
    resident._tiles_key = None
    with torch.cuda.graph(torch.cuda.CUDAGraph()):
        here = torch.zeros(1, device="cuda")
        with pytest.raises(_abi.GtmError, match="tiles of this model's sizes"):
            tm.score_device(sets[2])
    want_new = tm.score(new)
    # resident and done: captured, on another stream than the default one where it was made
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = tm.score_device(new)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy().reshape(want_new.shape), want_new)
        assert np.array_equal(tm.score(sets[0]), want[0])

    class Unfinished:
        def query(self):
            return False

    tm._test_graphs._made = Unfinished()
    with torch.cuda.graph(torch.cuda.CUDAGraph()):
        here = torch.zeros(1, device="cuda")
        with pytest.raises(_abi.GtmError, match="on its way"):
            tm.score_device(new)
    assert np.array_equal(tm.score(new), want_new)


def test_what_is_recorded_in_a_graph_does_not_stand_for_the_upload():
    """An event recorded under capture tells nothing about the upload, and cannot be asked."""
    import torch

    tm, sets, want = _model_and_sets()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        tm.score(sets[1])
        tm._test_graphs._made = None  # as after a call that failed between the tiles and its end
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        graph.capture_begin()
        out = tm.score_device(sets[1])
        graph.capture_end()
    assert tm._test_graphs._made is None
    for _ in range(3):
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy().reshape(want[1].shape), want[1])
        assert np.array_equal(tm.score(sets[0]), want[0])
