"""Brings the arrays of a ``Graphs`` object to the device.

Where the reference copies every array as it is (tm.py:528-555, 759-784), the
arrays cross the bus in the packed form of csrc/pack.c - the positive halves of
the literal words, numbers at the width they need - through pinned memory, and
one launch (``gtm_unpack_graphs``) makes the arrays the kernels index of it.
A pageable copy is a staged copy by one thread inside the driver; here all
threads pack, and packing one piece overlaps with the transfer of the last.
"""

import ctypes

import numpy as np
import torch

from . import _abi
from .graphs import _native_encoder

# Packed bytes per transfer.  A set that fits one takes one copy; larger ones are cut so that a piece is packed
# while the one before it is on its way.
PIECE_BYTES = 2 << 20
PIECES = 3

_ARRAYS = ("X", "node_type", "number_of_graph_node_edges", "edge", "node_index", "edge_index", "number_of_graph_nodes")


class _Image:
    """The packed image on the device, filled from the host piece by piece through a ring of pinned buffers."""

    def __init__(self, nbytes, largest_item, device):
        self.device = torch.empty(nbytes, dtype=torch.uint8, device=device)
        # (one size for whatever data set: pinned memory of a new size takes 100 to 200 us the first time)
        self.piece = max(PIECE_BYTES, 16 * largest_item)
        self.ring = []  # [pinned buffer, event after its last transfer]
        self.turn = 0
        self.open = None  # the ring's entry that is being filled
        self.sent = self.filled = 0  # bytes of the image that are on their way / in the open piece

    def _buffer(self):
        if self.open is None:
            if self.turn < PIECES:
                try:
                    buffer = torch.empty(self.piece, dtype=torch.uint8, pin_memory=True)
                except RuntimeError as e:
                    raise torch.OutOfMemoryError("no pinned memory") from e
                self.ring.append((buffer, torch.cuda.Event()))
            self.open = self.ring[self.turn % PIECES]
            if self.turn >= PIECES:
                self.open[1].synchronize()
            self.turn += 1
        return self.open[0]

    def flush(self):
        if self.filled:
            buffer, done = self.open
            self.device[self.sent:self.sent + self.filled].copy_(buffer[:self.filled], non_blocking=True)
            if self.filled < self.device.numel():
                done.record()
            self.sent += self.filled
            self.filled = 0
            self.open = None

    def append(self, items, item_bytes, pack):
        """``pack(first, count, address)`` writes the packed form of ``count`` items.  Returns the part's place in
        the image, or None when a call says (by a true value) that the items have no such form."""
        place, done = self.sent + self.filled, 0
        while done < items:
            count = min(items - done, (self.piece - self.filled) // item_bytes)
            if count < items - done:
                count &= ~15  # a cut piece ends, like a part, on a multiple of 16 bytes
            if count == 0:
                self.flush()
                continue
            if pack(done, count, self._buffer().data_ptr() + self.filled):
                return None
            self.filled += count * item_bytes
            done += count
        self.filled = _align(self.filled)
        return place


def _align(n):
    return (n + 15) & ~15


def upload(graphs, device):
    """(tensors by name, True when every negated literal is the complement of its positive one and every graph has
    a node) or None when the arrays are not as the packer addresses them, or when there is no room for the packed image
    beside them (half as much again) or for pinned memory.  Then they are copied as they are."""
    lib = _native_encoder()
    arrays = {name: getattr(graphs, name) for name in _ARRAYS}
    if lib is None or any(
        not isinstance(a, np.ndarray) or a.dtype != np.uint32 or not a.flags.c_contiguous for a in arrays.values()
    ):
        return None
    X, edge = arrays["X"], arrays["edge"]
    N, G, E = X.shape[0], arrays["number_of_graph_nodes"].shape[0], edge.shape[0]
    hv = int(graphs.hypervector_size)
    if X.ndim != 2 or N == 0 or G == 0 or hv < 1 or X.shape[1] != (2 * hv - 1) // 32 + 1:
        return None
    if edge.shape != (E, 2) or any(arrays[n].shape != (N,) for n in ("node_type", "number_of_graph_node_edges", "edge_index")) \
            or arrays["node_index"].shape != (G,):
        return None
    try:
        return _upload(lib, arrays, hv, device)
    except torch.OutOfMemoryError:
        pass  # (and the image is given back here, with the exception)
    return None


def _upload(lib, arrays, hv, device):
    X, edge = arrays["X"], arrays["edge"]
    N, G, E = X.shape[0], arrays["number_of_graph_nodes"].shape[0], edge.shape[0]
    at = {name: a.ctypes.data for name, a in arrays.items()}
    LA, words = X.shape[1], (hv + 31) // 32
    plan = np.empty(8, dtype=np.uint32)
    edge_start = np.empty(G, dtype=np.uint32)
    lib.gtm_pack_plan(at["node_type"], at["number_of_graph_node_edges"], at["edge_index"], at["node_index"],
                      at["number_of_graph_nodes"], at["edge"], N, E, G, plan.ctypes.data, edge_start.ctypes.data)
    type_bytes, type_value, degree_bytes, degree_value, follows, edge_bytes, some_empty = (int(v) for v in plan[:7])
    for positive in (True, False):
        row_bytes = 4 * (words if positive else LA)
        parts = [
            ("rows", N, row_bytes, None),
            ("types", N, type_bytes, at["node_type"]),
            ("degrees", N, degree_bytes, at["number_of_graph_node_edges"]),
            ("first_edges", G if follows else N, 4, edge_start.ctypes.data if follows else at["edge_index"]),
            ("edges", 2 * E, edge_bytes, at["edge"]),
            ("first_nodes", G, 4, at["node_index"]),
            ("node_counts", G, 4, at["number_of_graph_nodes"]),
        ]
        image = _Image(sum(_align(n * width) for _, n, width, _ in parts), row_bytes, device)
        packed = _abi.PackedGraphs()
        base = image.device.data_ptr()
        whole = True
        for name, n, width, source in parts:
            if n * width == 0:
                continue
            if name != "rows":
                place = image.append(n, width, lambda first, count, to: lib.gtm_pack_numbers(source + 4 * first, count, width, to))
            elif positive:
                place = image.append(n, width, lambda first, count, to: lib.gtm_pack_rows(at["X"] + 4 * LA * first, count, LA, hv, to))
            else:
                place = image.append(n, width, lambda first, count, to: lib.gtm_pack_numbers(at["X"] + 4 * LA * first, count * LA, 4, to))
            if place is None:
                whole = False  # some literal words do not follow from the positive ones: all of them are sent
                break
            setattr(packed, name, base + place)
        if whole:
            image.flush()
            break
    sizes = [(name, arrays[name].size) for name in _ARRAYS]
    everything = torch.empty(sum(-(-n // 64) * 64 for _, n in sizes), dtype=torch.int32, device=device)
    tensors, offset = {}, 0
    for name, n in sizes:
        tensors[name] = everything[offset:offset + n]
        if n:
            setattr(packed, name, everything.data_ptr() + 4 * offset)
        offset += -(-n // 64) * 64
    packed.total_nodes, packed.total_edges, packed.number_of_graphs = N, E, G
    packed.literal_words, packed.hypervector_size, packed.rows_positive = LA, hv, int(positive)
    packed.type_bytes, packed.type_value = type_bytes, type_value
    packed.degree_bytes, packed.degree_value = degree_bytes, degree_value
    packed.edge_bytes, packed.index_follows = edge_bytes, follows
    _abi.call("gtm_unpack_graphs", ctypes.byref(packed), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    # (the image is given back to the allocator of this stream with the launch that reads it already enqueued)
    return tensors, positive and not some_empty
