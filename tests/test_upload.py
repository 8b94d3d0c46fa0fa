"""Data sets packed for the bus (csrc/pack.c, upload.py) and unpacked on the device (gtm_unpack_graphs)."""

import copy

import numpy as np
import pytest

from tests import helpers

ARRAYS = ("X", "node_type", "number_of_graph_node_edges", "edge", "node_index", "edge_index", "number_of_graph_nodes")


def graphs_of(hv, **kwargs):
    args = dict(n_graphs=20, max_nodes=30, hv_size=hv, min_nodes=0, edge_types=("a", "b"), node_types=("x", "y"))
    args.update(kwargs)
    return helpers.random_graphs(hv, **args)


@pytest.mark.parametrize("hv", [10, 16, 31, 32, 33, 50, 64, 96, 200, 1000])
def test_rows_are_packed_and_any_flipped_bit_is_seen(hv):
    from graphtsetlinmachine_amd.graphs import _native_encoder

    lib = _native_encoder()
    X = graphs_of(hv).X
    N, LA = X.shape
    out = np.full((N, (hv + 31) // 32), 0x5A5A5A5A, dtype=np.uint32)
    pack = lambda x: lib.gtm_pack_rows(x.ctypes.data, N, LA, hv, out.ctypes.data)
    assert pack(X) == 0
    bits = lambda a: np.unpackbits(a.view(np.uint8), axis=1, bitorder="little")
    assert np.array_equal(bits(out)[:, :hv], bits(X)[:, :hv]) and not bits(out)[:, hv:].any()
    for row, bit in ((0, 0), (N - 1, hv - 1), (N // 2, hv), (1, 2 * hv - 1), (2, LA * 32 - 1)):
        broken = X.copy()
        broken[row, bit // 32] ^= np.uint32(1 << (bit % 32))
        assert pack(broken) == 1, (row, bit)


def broken_copies(g):
    """Data sets whose public arrays a caller has changed so that some of them no longer follow from less."""
    yield g, True
    x = copy.deepcopy(g)
    x.X[-1, 0] ^= np.uint32(1)
    yield x, False
    x = copy.deepcopy(g)
    if x.edge.size:
        x.edge_index[-1] += np.uint32(1)
        x.edge[0, 1] = 70000
        x.node_type[-1], x.number_of_graph_node_edges[-1] = 300, 256
    yield x, True


@pytest.mark.gpu
@pytest.mark.parametrize("piece", [128, 4096, 2 << 20])
@pytest.mark.parametrize("shape", [
    dict(hv=32), dict(hv=50, node_types=("x",), max_degree=0), dict(hv=96, min_nodes=1), dict(hv=200),
    dict(hv=64, n_graphs=3, max_nodes=1), dict(hv=1000, n_graphs=70, max_nodes=130),
], ids=lambda s: "hv%d" % s["hv"])
def test_the_device_holds_the_arrays_as_they_are(shape, piece, monkeypatch):
    import torch

    from graphtsetlinmachine_amd import upload

    monkeypatch.setattr(upload, "PIECE_BYTES", piece)
    args = dict(shape)
    for g, follows in broken_copies(graphs_of(args.pop("hv"), **args)):
        tensors, complementary = upload.upload(g, torch.device("cuda"))
        for name in ARRAYS:
            want = getattr(g, name)
            assert np.array_equal(tensors[name].cpu().numpy().view(np.uint32), want.reshape(-1)), name
        assert complementary == (follows and bool((g.number_of_graph_nodes > 0).all()))
    g.X = np.asfortranarray(g.X)
    assert upload.upload(g, torch.device("cuda")) is None


@pytest.mark.parametrize("node_index, node_counts", [
    ([0, 400000000], [400000000, 0]),              # the chain of graphs holds, far past the nodes
    ([0, 1000000, 1000002], [2, 2, 2]),            # a break, and the chain goes on behind it
    ([0, 4294967290], [4294967290, 12]),           # sums past 32 bits
    ([7, 3], [3, 7]),                              # graphs in another order
], ids=["past_the_nodes", "break", "wrap", "order"])
def test_graphs_that_do_not_follow_one_another_are_only_looked_at_inside_the_arrays(node_index, node_counts):
    from graphtsetlinmachine_amd.graphs import _native_encoder

    N = 10
    u32 = lambda values: np.array(values, dtype=np.uint32)
    node_type, degree, edge_index = u32([0] * N), u32([1] * N), u32(range(N))
    first, count, edge = u32(node_index), u32(node_counts), np.zeros((N, 2), dtype=np.uint32)
    plan, start = np.full(8, 0x5A5A5A5A, dtype=np.uint32), np.zeros(len(first), dtype=np.uint32)
    _native_encoder().gtm_pack_plan(*(a.ctypes.data for a in (node_type, degree, edge_index, first, count, edge)), N, N, len(first),
                                    plan.ctypes.data, start.ctypes.data)
    assert list(plan[:3]) == [0, 0, 0] and plan[4] == 0  # all types and degrees alike; first edges do not follow


@pytest.mark.parametrize("sizes, follows", [
    ([1024], 1), ([1025], 0), ([1000000], 0), ([5000] + [3] * 500, 0), ([2000] * 63, 0), ([2000] * 64, 1), ([1024, 0, 7], 1),
], ids=["1024", "1025", "million", "one_large_among_small", "63_of_2000", "64_of_2000", "ragged"])
def test_first_edges_are_summed_on_the_device_where_graphs_are_many_or_small(sizes, follows):
    from graphtsetlinmachine_amd.graphs import _native_encoder

    count = np.array(sizes, dtype=np.uint32)
    first = (np.cumsum(count) - count).astype(np.uint32)
    N, G = int(count.sum()), len(count)
    zeros, edge = np.zeros(N, dtype=np.uint32), np.zeros((1, 2), dtype=np.uint32)
    plan, start = np.zeros(8, dtype=np.uint32), np.zeros(G, dtype=np.uint32)
    _native_encoder().gtm_pack_plan(*(a.ctypes.data for a in (zeros, zeros, zeros, first, count, edge)), N, 0, G, plan.ctypes.data,
                                    start.ctypes.data)
    assert plan[4] == follows


def _refusing(monkeypatch, is_refused):
    import torch

    empty = torch.empty

    def refuse(*size, **kwargs):
        if is_refused(kwargs):
            raise torch.OutOfMemoryError("no room")
        return empty(*size, **kwargs)

    monkeypatch.setattr(torch, "empty", refuse)


@pytest.mark.parametrize("refused", [lambda k: True, lambda k: False], ids=["image", "pinned"])
def test_without_room_the_arrays_are_left_to_plain_copies(refused, monkeypatch):
    import torch

    from graphtsetlinmachine_amd import upload

    _refusing(monkeypatch, refused)
    if torch.cuda.is_available():
        _refusing(monkeypatch, lambda k: refused(k) or k.get("pin_memory"))  # (without a device there is no pinned memory)
    assert upload.upload(graphs_of(32), torch.device("cpu")) is None


@pytest.mark.gpu
@pytest.mark.parametrize("piece", [128, 2 << 20])
@pytest.mark.parametrize("refused", [
    lambda k: k.get("dtype") is not None and str(k["dtype"]) == "torch.int32", lambda k: k.get("pin_memory")], ids=["arrays", "pinned"])
def test_without_room_the_device_still_holds_the_arrays(refused, piece, monkeypatch):
    from graphtsetlinmachine_amd import upload
    from graphtsetlinmachine_amd.tm import _DeviceGraphs

    g = graphs_of(64, n_graphs=70, max_nodes=130)
    monkeypatch.setattr(upload, "PIECE_BYTES", piece)
    with monkeypatch.context() as m:
        _refusing(m, refused)
        dg = _DeviceGraphs(g)
    assert dg._complementary is None  # (plain copies: not looked at)
    for name in ARRAYS:
        assert np.array_equal(dg.tensors[name].cpu().numpy().view(np.uint32), getattr(g, name).reshape(-1)), name


@pytest.mark.gpu
def test_small_data_sets_of_any_size_share_their_pinned_memory(monkeypatch):
    import torch

    from graphtsetlinmachine_amd import upload

    asked, empty = set(), torch.empty

    def watch(*size, **kwargs):
        if kwargs.get("pin_memory"):
            asked.add(size)
        return empty(*size, **kwargs)

    monkeypatch.setattr(torch, "empty", watch)
    for n in (1, 3, 20, 150):
        upload.upload(graphs_of(64, n_graphs=n), torch.device("cuda"))
    assert asked == {(upload.PIECE_BYTES,)}


def test_the_packer_keeps_no_data_of_its_own(tmp_path):
    """Calls from several threads run side by side (ctypes releases the interpreter lock): no static that one writes and another reads."""
    import shutil
    import subprocess

    from graphtsetlinmachine_amd import build

    if not (shutil.which("gcc") and shutil.which("nm")):
        pytest.skip("needs gcc and nm")
    source = [s for s in build.ENCODER_SOURCES if s.endswith("pack.c")][0]
    subprocess.run(["gcc", "-O3", "-fopenmp", "-fPIC", "-c", "-o", str(tmp_path / "pack.o"), source], check=True)
    symbols = subprocess.run(["nm", str(tmp_path / "pack.o")], check=True, capture_output=True, text=True).stdout.splitlines()
    assert any(line.endswith(" T gtm_unpack_outputs") for line in symbols)
    assert not [line for line in symbols if line.split()[-2] in "bBdDC"]
