"""Clause outputs on their way to the host as bits, and per node from the truth rows: the same arrays whichever way they take."""

import ctypes

import numpy as np
import pytest

from oracle import gtm_oracle as o
from tests import helpers


@pytest.mark.parametrize("n", [1, 31, 32, 33, 1024, 4097 * 32 + 5])
def test_bits_become_outputs_again(n):
    from graphtsetlinmachine_amd.graphs import _native_encoder

    want = np.random.default_rng(n).integers(0, 2, size=n).astype(np.int32)
    bits = np.packbits(np.pad(want, (0, -n % 32)).astype(np.uint8), bitorder="little")
    out = np.full(n + 1, 7, dtype=np.int32)
    _native_encoder().gtm_unpack_outputs(bits.ctypes.data, n, out.ctypes.data)
    assert np.array_equal(out[:n], want) and out[n] == 7


@pytest.mark.parametrize("n", [0, 1, 4095, 4096, 4097, 8192, 70000, 1 << 20])
def test_touching_pages_stays_in_the_array(n):
    from graphtsetlinmachine_amd.graphs import _native_encoder

    array = np.full(n + 8, 7, dtype=np.uint8)
    _native_encoder().gtm_touch_pages(array.ctypes.data, n)
    want = np.full(n + 8, 7, dtype=np.uint8)
    want[:n:4096] = 0
    assert np.array_equal(array, want)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 63, 64, 65, 1023, 2048 * 1024 + 77])  # the last: more than one turn of the largest grid
def test_outputs_become_bits(n):
    import torch

    from graphtsetlinmachine_amd import _abi
    from graphtsetlinmachine_amd.tm import _ptr, _stream

    values = np.random.default_rng(n).integers(-1, 2, size=n).astype(np.int32)
    bits = torch.full(((n + 31) // 32 + 1,), 0x5A5A5A5A, dtype=torch.int32, device="cuda")
    outputs = torch.from_numpy(values).cuda()
    _abi.call("gtm_pack_outputs", _ptr(outputs), n, _ptr(bits), _stream())
    got = bits.cpu().numpy()
    assert got[-1] == 0x5A5A5A5A
    assert np.array_equal(got[:-1].view(np.uint8), np.packbits(np.pad(values != 0, (0, -n % 32)), bitorder="little"))


@pytest.mark.gpu
@pytest.mark.parametrize("sizes,clauses", [([1], 3), ([1, 1, 1], 17), ([2, 1, 2, 0], 40), ([33, 7, 0, 20], 501), ([130, 64, 97], 300), ([700, 841], 40)],
                         ids=str)
@pytest.mark.parametrize("depth", [1, 2])
def test_outputs_whichever_way_they_take(sizes, clauses, depth, monkeypatch):
    from graphtsetlinmachine_amd import tm as tm_module

    graphs = helpers.random_graphs(clauses, n_graphs=3 * len(sizes), sizes=sizes * 3, hv_size=40, max_degree=2)
    tm = tm_module.MultiClassGraphTsetlinMachine(clauses, 30, 2.0, depth=depth, message_size=64, message_bits=2, seed=3)
    tm.fit(graphs, np.arange(3 * len(sizes)) % 3, epochs=2)
    cfg = helpers.oracle_config(graphs, classes=3, clauses=clauses, message_size=64, T=30)
    state = tm.get_state()
    model = o.new_model(cfg, depth, 2.0, tm.hypervectors, seed=3)
    model.ta_state = state[0].reshape(clauses, -1, 8)
    model.clause_weights = state[1].reshape(3, clauses)
    model.message_ta_state = [b.reshape(clauses, -1, 8) for b in state.message_ta_state]
    want, want_sums = o.transform(model, graphs)
    want_wide, _ = o.transform(model, graphs, nodewise=True)
    native, calls = tm_module._native_encoder(), []
    waited = tm_module.torch.cuda.Stream.synchronize

    class Recorder:
        def __getattr__(self, name):
            return lambda *args: (calls.append(name), getattr(native, name)(*args))[1]

    monkeypatch.setattr(tm_module, "_native_encoder", lambda: Recorder())
    monkeypatch.setattr(tm_module.torch.cuda.Stream, "synchronize", lambda stream: (calls.append("wait"), waited(stream))[1])
    for bits_from, pinned in ((0, 1 << 24), (0, 0), (1 << 40, 0)):
        monkeypatch.setattr(tm_module, "OUTPUTS_AS_BITS", bits_from)
        monkeypatch.setattr(tm_module, "PINNED_RESULT", pinned)
        calls.clear()
        got, sums = tm.transform(graphs)
        # (a new array's pages are made while the device works, not after the wait)
        seen = [c for c in calls if c in ("gtm_touch_pages", "wait", "gtm_unpack_outputs")]
        want_calls = [] if bits_from else ["gtm_touch_pages"] + ["wait"] * bool(pinned) + ["gtm_unpack_outputs"]
        assert seen[-len(want_calls):] == want_calls if want_calls else "gtm_unpack_outputs" not in seen
        assert got.dtype == sums.dtype == np.int32 and got.flags.writeable and sums.flags.writeable
        assert np.array_equal(got, want) and np.array_equal(sums, want_sums)
        got, sums = tm.transform_nodewise(graphs)
        assert got.dtype == np.int32 and np.array_equal(got, want_wide) and np.array_equal(sums, want_sums)
