"""Whole-network packed inference: a frozen dense network (LogicLayer ... GroupSum) evaluated
in one kernel launch per batch of packed samples (csrc/packed_net.hip).

This is the cross-module fusion of the layer-by-layer packed path (LogicLayer.forward on a
PackBitsTensor, then GroupSum): the counts are identical, but no intermediate layer is written
to HBM.  It plays the role of the compiled whole-network evaluators of the reference lineage
(third_party/convlogic_source_code/src/difflogic/compiled_model.py:159-242), built from the
same argmax-slot semantics as compactlogic/compactlogic.py:120-130.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from . import _capi
from . import timing
from . import convlogic_hip as _cl
from . import difflogic_hip as _dl
from . import packed_circuit as _pc
from .layers import ConvLayer, GroupSum, LogicLayer, PackBitsTensor
from .treelogic import ConvLogicLayer


def _limits():
    nl, rows = ctypes.c_int64(0), ctypes.c_int64(0)
    _capi.call("cl_packed_network_limits", ctypes.byref(nl), ctypes.byref(rows))
    return nl.value, rows.value


# LDS geometry of gfx950 as the fused kernel uses it (measured with 64-lane ds_read_b32
# patterns and SQ_LDS_BANK_CONFLICT): a read instruction is served one half-wave (32 lanes) at
# a time, and the lanes of a half-wave conflict when their words share word % 32.  The lanes of
# one half-wave read the rows of 32 consecutive positions of the layer being computed.
_LDS_BANKS = 32
_HALF_WAVE = 32


def _i32(a):
    return np.ascontiguousarray(a, dtype=np.int32)


def _layout(ka, kb, fa, fb, rows: int, class_size: int) -> np.ndarray:
    P = ctypes.POINTER(ctypes.c_int32)
    ka, kb = _i32(ka), _i32(kb)
    pos = np.empty(int(rows), dtype=np.int32)
    fa_ = None if fa is None else _i32(fa)
    fb_ = None if fb is None else _i32(fb)
    _capi.call("cl_packed_bank_layout", ka.ctypes.data_as(P), kb.ctypes.data_as(P),
               None if fa_ is None else fa_.ctypes.data_as(P),
               None if fb_ is None else fb_.ctypes.data_as(P), int(rows), int(class_size),
               pos.ctypes.data_as(P))
    return pos.astype(np.int64)


def bank_aware_positions(pos_a: np.ndarray, pos_b: np.ndarray, rows: int,
                         fan_a: np.ndarray | None = None,
                         fan_b: np.ndarray | None = None) -> np.ndarray:
    """Positions (LDS words, a permutation of 0..rows-1) for the gates of one layer whose
    inputs sit at words pos_a / pos_b of the previous layer (cl_packed_bank_layout): blocks of
    32 consecutive positions (one half-wave of the kernel's row reads) that read their a rows
    from 32 distinct banks and their b rows from 32 distinct banks, from an edge colouring of
    the (bank a, bank b) multigraph with one colour per block.  Inside a block the position is
    free for this layer; with the next layer's fan-outs of these rows (fan_a: reads as operand
    a, fan_b: as operand b) it is chosen to level the next layer's bank degrees, which is what
    lets that layer's colouring avoid conflicts.  Deterministic."""
    return _layout(np.asarray(pos_a) % _LDS_BANKS, np.asarray(pos_b) % _LDS_BANKS, fan_a, fan_b,
                   rows, 0)


def bank_aware_positions_grouped(pos_a: np.ndarray, pos_b: np.ndarray, rows: int,
                                 group_size: int) -> np.ndarray:
    """bank_aware_positions for the last layer, whose rows must stay in their class: gate o
    (class o // group_size) is placed inside [class * group_size, (class + 1) * group_size).
    Deterministic."""
    return _layout(np.asarray(pos_a) % _LDS_BANKS, np.asarray(pos_b) % _LDS_BANKS, None, None,
                   rows, group_size)


# the fused kernel stages each 32-sample column of its input in LDS: at most _LDS_INPUT_ROWS
# input rows (four per thread).  Gathering one word of every input row per column from a wider
# input is bound by L2 capacity (the rows' lines of 32 columns must stay resident), and a
# kernel that did so measured 3.7-7x slower than the layer path.
_LDS_INPUT_ROWS = 4096


def _fusable(in_rows: int, outs: list, max_layers: int, max_rows: int) -> bool:
    """Whether cl_packed_network takes dense layers of widths `outs` on `in_rows` inputs."""
    return (bool(outs) and len(outs) <= max_layers and in_rows <= _LDS_INPUT_ROWS
            and max(outs) <= max_rows)


def columns_layout(rows: list) -> dict | None:
    """LDS placement of the wide-input fused pass for layer widths `rows` (input first), or
    None when it does not apply (cl_packed_network_columns_layout): in_words (LDS words per
    input column), split and hold_base (row p of the first layer is word base[0] + p below
    split, else hold_base + p - split) and base (row p of layer l >= 1 is word base[l] + p)."""
    n = len(rows) - 1
    if n < 1 or n > _limits()[0]:
        return None
    arr = (ctypes.c_int64 * len(rows))(*[int(r) for r in rows])
    applies, in_words, split, hold = (ctypes.c_int64() for _ in range(4))
    base = (ctypes.c_int64 * n)()
    _capi.call("cl_packed_network_columns_layout", arr, n, ctypes.byref(applies),
               ctypes.byref(in_words), ctypes.byref(split), ctypes.byref(hold), base)
    if not applies.value:
        return None
    return {"in_words": in_words.value, "split": split.value, "hold_base": hold.value,
            "base": list(base)}


def producer_order(tabs: list, in_rows: int) -> np.ndarray:
    """Order in which the column producer evaluates its rows (int32, a permutation): rows
    sorted by the sorted tuple of the blocks (in_rows // 16 rows each) of the input rows they
    read, ties in row order.  Rows reading the same input blocks then run together, so the
    input words of a column tile they need stay in one XCD's L2.  tabs: the (ia, ib) index
    arrays of the producer's layers (one, or two composed, the second reading the first's
    rows); a negative or out-of-range index reads nothing."""
    blk = max(1, in_rows // 16)
    none = in_rows // blk + 1

    def blocks(rows, n):
        ok = (rows >= 0) & (rows < n)
        return ok, np.where(ok, rows, 0)

    if len(tabs) == 1:
        ia, ib = tabs[0]
        cols = []
        for r in (ia, ib):
            ok, rr = blocks(r, in_rows)
            cols.append(np.where(ok, rr // blk, none))
    else:
        (ia1, ib1), (ia2, ib2) = tabs
        mid = ia1.size
        cols = []
        for r2 in (ia2, ib2):
            ok2, p = blocks(r2, mid)
            for r1 in (ia1, ib1):
                ok1, rr = blocks(r1[p], in_rows)
                cols.append(np.where(ok2 & ok1, rr // blk, none))
    key = np.sort(np.stack(cols, 1), axis=1)
    n = key.shape[0]
    return np.lexsort((np.arange(n),) + tuple(key[:, j] for j in reversed(range(key.shape[1])))
                      ).astype(np.int32)


def _tree_front(prefix: list) -> list | None:
    """The complete ConvLogicLayers that make up `prefix` (Flatten modules pass a PackBitsTensor
    through unchanged); None when it holds anything else or nothing."""
    blocks = [m for m in prefix if type(m) is not torch.nn.Flatten]
    ok = all(type(m) is ConvLogicLayer and m.complete for m in blocks)
    return blocks if blocks and ok else None


def tree_columns_layout(blocks: list, rows: int) -> tuple | None:
    """(geometry array, output rows, table words) of cl_tree_columns for the blocks on a square
    input of `rows` features, or None when the pass does not take them
    (cl_tree_columns_layout)."""
    if rows % blocks[0].in_channels:
        return None
    h = w = math.isqrt(rows // blocks[0].in_channels)
    if h * w * blocks[0].in_channels != rows:
        return None
    geo = []
    for m in blocks:
        (sh, sw), (ph, pw), (kh, kw) = m.stride, m.padding, m.kernel
        geo += [m.in_channels, h, w, m.out_channels, sh, sw, ph, pw, kh, kw]
        h, w = ((h + 2 * ph - kh) // sh + 1) // 2, ((w + 2 * pw - kw) // sw + 1) // 2
    arr = (ctypes.c_int64 * len(geo))(*geo)
    out = [ctypes.c_int64(0) for _ in range(4)]
    _capi.call("cl_tree_columns_layout", arr, len(blocks), *[ctypes.byref(v) for v in out])
    return (arr, out[2].value, out[3].value) if out[0].value else None


def tree_columns_from(blocks: list, rows: int) -> float:
    """Number of 32-sample columns from which cl_tree_columns is faster than the blocks one by one
    on a square input of `rows` features (inf: never).  The column pass turns every input row to
    columns and gives a wave a channel of 64 positions (`whole` rows, channels rounded up to the
    sixteen waves; `others`: a lane per position); the row kernels read the rows that are tapped
    and cost a launch per block.  Measured, columns / rows, for 64 K and 1 M samples: 9 x 32 x 32
    -> 256 -> 512 channels 0.75, 0.59; -> 64 -> 128 1.37, 0.86; -> 16 2.2, 1.09; 2 x 16 x 16 -> 64
    0.94, 0.54, -> 17 1.29, 1.11; 64 x 16 x 16 -> 64 2.6, 1.36; 3 x 12 x 12 -> 10 -> 12 (36 and 9
    positions) 1.08, 1.97."""
    h = w = math.isqrt(rows // blocks[0].in_channels)
    whole = waves = others = 0
    for m in blocks:
        (sh, sw), (ph, pw), (kh, kw) = m.stride, m.padding, m.kernel
        h, w = ((h + 2 * ph - kh) // sh + 1) // 2, ((w + 2 * pw - kw) // sw + 1) // 2
        if h * w % 64:
            others += m.out_channels * h * w
        else:
            whole += m.out_channels * h * w
            waves += -(-m.out_channels // 16) * 16 * h * w
    if 5 * whole < 2 * waves + others + rows + 1200:
        return math.inf
    return 2 ** 24 / whole


def _table_layer_before(body: list, j: int):
    """Index of the module before body[j] (Flatten modules pass a PackBitsTensor through
    unchanged) when it is a packed layer from index tables (ConvLayer or LogicLayer); else
    None."""
    j -= 1
    while j >= 0 and type(body[j]) is torch.nn.Flatten:
        j -= 1
    if j < 0 or type(body[j]) not in (ConvLayer, LogicLayer):
        return None
    return j


def _column_words(layout: dict, layer: int, pos: np.ndarray) -> np.ndarray:
    """LDS words of layer `layer`'s rows at positions pos under a columns_layout (banks as the
    positions': every base is a multiple of 32 words)."""
    if layer == 0:
        return np.where(pos < layout["split"], layout["base"][0] + pos,
                        layout["hold_base"] + pos - layout["split"])
    return layout["base"][layer] + pos


def _on_host(tabs: list) -> list:
    return [tuple(t.cpu().numpy().astype(np.int64) for t in tab) for tab in tabs]


# Bytes of a producer's packed input up to which its circuit reads the rows as they lie, a word
# pair per row: they stay in the Infinity Cache then, and a launch is saved (two convolutions of
# 9 x 32 x 32 and 2 x 16000, rows / columns: 23 / 32 us for 64 samples, 120 / 133 for 128 K, 274 /
# 284 for 256 K (302 MB), 974 / 875 for 768 K; one of 3 x 40 x 40 and 3500 194 / 219 for 512 K
# (315 MB), 376 / 345 for 768 K).
_ROWS_IN_CACHE = 256 << 20


class _Circuit:
    """A tail's pruned circuit (packed_circuit.build) on the device."""

    @classmethod
    def of(cls, layers: list, in_rows: int, k: int, device, row_slots: int | None = None):
        """The circuit of layers [(a, b, opcode), ...], or None where it does not fit or pay
        (packed_circuit.build)."""
        plan = _pc.build(_pc.fold(layers, in_rows), k, row_slots)
        return None if plan is None else cls(plan, in_rows, device)

    def __init__(self, plan: dict, in_rows: int, device):
        self.in_rows, self.k = in_rows, plan["shape"][5]
        self.shape = (ctypes.c_int64 * 7)(*plan["shape"])
        # one buffer, its tables at 16-byte offsets; their addresses are computed when it moves
        # (a copy of this object has a buffer of its own), not per call
        parts, self.offsets, end = [], [], 0
        self.base, self.at = None, ()
        for name in ("ent", "ops", "dst", "in", "cnt", "ones"):
            raw = plan[name].reshape(-1).view(np.uint8)
            parts.append(np.pad(raw, (0, -raw.size % 16)))
            self.offsets.append(end)
            end += parts[-1].size
        self.tables = torch.as_tensor(np.concatenate(parts).view(np.int32), device=device)
        self.gates = plan["gates"]

    def __call__(self, words, cols: int, columns_major: bool, in_words: int, n: int):
        counts = torch.empty((n, self.k), dtype=torch.int32, device=words.device)
        base = self.tables.data_ptr()
        if base != self.base:
            self.at, self.base = tuple(base + o for o in self.offsets), base
        at = self.at
        with _dl.on_device_of(words):
            timing.timed(f"cl_packed_circuit[{self.in_rows}]", lambda: _capi.call(
                "cl_packed_circuit", words.data_ptr(), cols, int(columns_major), in_words, n,
                self.shape, *at, counts.data_ptr(),
                _dl.stream_of(words)))
        return counts


class PackedNetwork:
    """Fused packed evaluator of `model` (frozen or in eval mode; each neuron uses its argmax
    slot `w`), ending in a GroupSum.  Call it with a PackBitsTensor of the network's input (or
    its [features, words] tensor) to get int32 class counts [samples, k].

    The longest tail of dense LogicLayers that the fused kernel takes (an input of at most
    4096 rows, widths within LDS) runs in one launch with every 32-sample column held in LDS;
    the modules before it (ConvLayers, ConvLogicLayers, wider dense layers, Flatten) run layer
    by layer on the packed kernels first.  A tail whose input is wider (cfg5's 25088 conv
    outputs) is fused when a ConvLayer or dense LogicLayer feeds it and its layers fit
    (columns_layout): that layer writes its output column-major
    (cl_eval_packed_indexed_columns) and the tail runs on those columns
    (cl_packed_network_columns).  When no tail qualifies every module runs layer by
    layer and the counts come from the group popcount.  A fused tail whose prefix is complete
    ConvLogicLayers alone takes its input column-major from them (cl_tree_columns: all blocks on
    one column in LDS) where that is the faster way (tree_columns_from).  Where it fits and pays
    (packed_circuit.build), a fused tail, or the whole network when the layers that
    write its columns come first, is reduced to the two-input gates that reach an output.
    The gate tables are built once here; rebuild after changing the model.  With `bank_aware` (default), each fused layer's rows
    are laid out in LDS by bank_aware_positions, so that the row reads of the kernel's
    half-waves hit distinct LDS banks; the counts do not depend on the layout.  With `prune`
    False every row of every layer is evaluated, as where no circuit fits.
    """

    def __init__(self, model, bank_aware: bool = True, prune: bool = True):
        mods = list(model)
        if not mods or not isinstance(mods[-1], GroupSum):
            raise ValueError("the network must end with a GroupSum")
        body = mods[:-1]
        if not body:
            raise ValueError("the network needs a layer before its GroupSum")
        max_layers, max_rows = _limits()
        self.k = int(mods[-1].k)
        # the fused tail: the longest run of trailing dense layers that the kernel takes
        first = len(body)
        while first > 0 and type(body[first - 1]) is LogicLayer:
            first -= 1
        start = next((j for j in range(first, len(body))
                      if _fusable(int(body[j].in_dim), [int(m.out_dim) for m in body[j:]],
                                  max_layers, max_rows)), len(body))
        # a tail whose input is too wide to stage row by row: its input comes column-major
        # from the packed layer before it (cl_eval_packed_indexed_columns)
        self.producer = None     # the layer (or pair of layers) writing the tail's columns
        self.layout = None
        if start != first and first < len(body):
            prod = _table_layer_before(body, first)
            rows = [int(body[first].in_dim)] + [int(m.out_dim) for m in body[first:]]
            layout = columns_layout(rows) if prod is not None else None
            if layout is not None:
                start, self.layout = first, layout
                # a table layer before the producer is composed into it: its rows are
                # computed where the producer reads them, never stored
                pre = _table_layer_before(body, prod)
                if pre is not None:
                    self.producer, self.prefix = (body[pre], body[prod]), body[:pre]
                else:
                    self.producer, self.prefix = (body[prod],), body[:prod]
        layers = body[start:]
        if self.producer is None:
            self.prefix = body[:start]
        if not layers:
            self.rows = None            # no fused tail: layer by layer, then the popcount
            self.device = None
            self.circuit = None
            return
        self.rows = [int(layers[0].in_dim)] + [int(m.out_dim) for m in layers]
        for i, (prev, m) in enumerate(zip(self.rows[:-1], layers)):
            if m.in_dim != prev:
                raise ValueError(f"layer {i} expects {m.in_dim} inputs, gets {prev}")
        if self.rows[-1] % self.k:
            raise ValueError(f"in_dim ({self.rows[-1]}) has to be divisible by k ({self.k}) "
                             "but it is not")
        # complete logic-tree blocks before the tail: they can hand it columns
        self.front = self.front_layout = self._front_from = None
        if self.producer is None:
            self.front = _tree_front(self.prefix)
            self.front_layout = columns_layout(self.rows) if self.front else None
            if self.front_layout is None:
                self.front = None
        wiring = []
        with torch.no_grad():
            for m in layers:
                w = getattr(m, "w", None)
                if w is None:
                    w = m.weights.argmax(-1)
                slot = w.to(torch.long).view(-1, 1)
                a = torch.gather(m.indices[0], 1, slot).view(-1).to(torch.int64)
                b = torch.gather(m.indices[1], 1, slot).view(-1).to(torch.int64)
                g = torch.gather(m.gate_sequence, 1, slot).view(-1).to(torch.int64) & 15
                if int(a.min()) < 0 or int(a.max()) >= m.in_dim or int(b.min()) < 0 or \
                        int(b.max()) >= m.in_dim:
                    raise IndexError("connection indices out of range")
                wiring.append((a.cpu().numpy(), b.cpu().numpy(), g.cpu().numpy()))
        self.device = layers[0].weights.device
        self._rows_host = (ctypes.c_int64 * len(self.rows))(*self.rows)
        self._wiring, self._bank_aware = wiring, bank_aware
        self._columns = None          # the producer's tables the row tables are laid out for
        self.tables = self.front_tables = self.col_order = None
        # the pruned circuit of the tail, where it fits, in place of the row tables: 22800
        # two-input gates of the 72000 of 784 -> 6 x 12000 take 1.51 ms for 4 M samples, all
        # rows 3.96; the 2 x 16000 tail of a logic-tree network 0.38 ms for 1 M, 0.66
        self.circuit = self.circuit_tabs = self._other_tabs = None
        if prune and bank_aware and self.k <= 1024 and not (self.producer and self.prefix):
            # with a producer, the layers that write the tail's columns and the tail as one
            # circuit: 29000 two-input gates of the 122600 rows of two convolutions of
            # 9 x 32 x 32 and 2 x 16000 take 1.29 ms for 1 M samples, producer and tail 2.47.
            # It stands for these tables of the layers: with others the call takes the row tables
            head = []
            if self.producer is not None:
                self.circuit_tabs = self._producer_tables()
                head = self._columns = _on_host(self.circuit_tabs)
            self.circuit = _Circuit.of(head + wiring,
                                       self._producer_rows() if head else self.rows[0], self.k,
                                       self.device, self._row_slots(head))
        if self.producer is not None and self._columns is None:
            self._columns = _on_host(self._producer_tables())
        if self.circuit is None:
            self._lay_out_rows()
        elif self.producer is None:
            self._wiring = None        # the tail does not change: its circuit is all it needs
        elif any(getattr(m, "w", None) is None for m in self.producer):
            # layers that may still train: under graph capture their winners are never known to
            # be the circuit's, and the row tables cannot be laid out there
            self._lay_out_rows()
        else:
            # the row tables, which take as long to lay out as the circuit, wait for the first
            # call with other tables; should that be under capture, the layers run one by one
            self._tail = [tuple(torch.as_tensor(t, dtype=d, device=self.device)
                                for t, d in zip(w, (torch.int32, torch.int32, torch.uint8)))
                          for w in wiring]

    def _row_slots(self, head: list) -> int:
        """Gate slots per thread in which the row tables are evaluated: the kernels give every
        layer of the tail the slots of its widest (their variants), a producer a row per slot."""
        widest = -(-max(self.rows[1:]) // 1024)
        per_layer = next((j for j in (1, 2, 4, 8, 12, 16) if widest <= j), widest)
        return per_layer * (len(self.rows) - 1) + sum(t[0].size for t in head) // 1024

    def _lay_out_rows(self) -> None:
        """The row tables: `tables` of the tail's layers (`front_tables`: for the column-major
        input that logic-tree blocks write) and `col_order`, the producer's row order."""
        prev_pos = np.arange(self.rows[0], dtype=np.int64)   # input rows stay in place
        lay, col_order = self.layout, None
        if self.producer is not None:
            # the producer writes its rows in producer_order; input row r of the tail is
            # then at position inv[r] of a column
            order = producer_order([t[:2] for t in self._columns], self._producer_rows())
            prev_pos = np.empty(self.rows[0], dtype=np.int64)
            prev_pos[order] = np.arange(self.rows[0], dtype=np.int64)
            col_order = torch.as_tensor(order, device=self.device)
        front_word = np.arange(self.rows[0], dtype=np.int64)  # LDS words in the columns
        entries, front_entries = [], []
        for i, (a, b, g) in enumerate(self._wiring):
            pa, pb = prev_pos[a], prev_pos[b]
            if not self._bank_aware:
                pos = np.arange(a.size, dtype=np.int64)
            elif i + 1 < len(self._wiring):
                na, nb = self._wiring[i + 1][:2]
                pos = bank_aware_positions(pa, pb, a.size, np.bincount(na, minlength=a.size),
                                           np.bincount(nb, minlength=a.size))
            else:  # class groups stay contiguous
                pos = bank_aware_positions_grouped(pa, pb, a.size, a.size // self.k)
            ent = np.empty(a.size, dtype=np.int64)
            if lay is None:
                ent[pos] = (pa * 4) | ((pb * 4) << 20) | (g << 40)   # LDS byte offsets
                prev_pos = pos
            else:
                ent[pos] = pa | (pb << 16) | (g << 32)               # LDS words
                prev_pos = _column_words(lay, i, pos)
            entries.append(ent)
            if self.front is not None:   # the same positions for the column-major input
                ent = np.empty(a.size, dtype=np.int64)
                ent[pos] = front_word[a] | (front_word[b] << 16) | (g << 32)
                front_word = _column_words(self.front_layout, i, pos)
                front_entries.append(ent)
        if front_entries:
            self.front_tables = torch.as_tensor(np.concatenate(front_entries), device=self.device)
        self.col_order = col_order
        # last: a call in another thread that finds it has the others
        self.tables = torch.as_tensor(np.concatenate(entries), device=self.device)

    def _circuit_holds(self, tabs: list) -> bool:
        """Whether the circuit stands for these tables of the producer.  Other table tensors than
        the last ones are compared by content, once (a synchronisation); under graph capture
        they count as other tables."""
        def same(old):
            return old is not None and all(t is c for tab, o in zip(tabs, old)
                                           for t, c in zip(tab, o))

        if same(self._other_tabs):
            return False
        if same(self.circuit_tabs):
            return True
        if tabs[0][0].is_cuda and torch.cuda.is_current_stream_capturing():
            return False
        if all(torch.equal(t, c) for tab, old in zip(tabs, self.circuit_tabs)
               for t, c in zip(tab, old)):
            self.circuit_tabs = tabs
            return True
        self._other_tabs = tabs
        return False

    def _layer_by_layer(self, words, tabs: list, n: int) -> torch.Tensor:
        """The producer and the tail one layer at a time (under graph capture, where the row
        tables cannot be laid out)."""
        for ia, ib, gate in [*tabs, *self._tail]:
            words = _cl.eval_packed_indexed(words, ia, ib, gate)
        pad = words.shape[1] * words.element_size() * 8 - n
        return _dl.groupbitsum(words, pad, self.k)

    def _producer_tables(self) -> list:
        """(ia, ib, gate) of the producer's layers as they are now."""
        tabs = []
        for m in self.producer:
            w = getattr(m, "w", None)
            tabs.append(m.packed_tables(m._argmax_slots() if w is None else w)[:3])
        return tabs

    def _producer_rows(self) -> int:
        m = self.producer[0]
        return m.in_dim if type(m) is LogicLayer else int(np.prod(m.in_shape))

    def __call__(self, x) -> torch.Tensor:
        if self.producer is not None:
            return self._call_columns(x)
        if self.prefix:
            counts = (self._call_front(x) if self.rows is not None and self.front
                      and self._front_pays(x) else None)
            if counts is not None:
                return counts
            if isinstance(x, PackBitsTensor):
                h = PackBitsTensor.from_packed(x.t, x.pad_len)   # the caller's object stays
            else:
                h = PackBitsTensor.from_packed(x)
            with torch.no_grad():
                for m in self.prefix:
                    h = m(h)
            if self.rows is None:
                return h.group_sum(self.k)
            x = h
        if isinstance(x, PackBitsTensor):
            words, n = x.t, x.num_samples
        else:
            words, n = x, x.shape[1] * x.element_size() * 8
        _dl._check(words, "x")
        if words.device != self.device:
            raise RuntimeError(f"x is on {words.device}, the network on {self.device}")
        if words.dim() != 2 or words.shape[0] != self.rows[0]:
            raise RuntimeError(f"x must be [{self.rows[0]}, words], got {tuple(words.shape)}")
        row_bytes = words.shape[1] * words.element_size()
        if self.circuit is not None:
            if row_bytes % 4:     # as cl_packed_network does
                raise _capi.CompactLogicError("packed rows must be a multiple of 4 bytes")
            return self.circuit(words, row_bytes // 4, False, 0, n)
        counts = torch.empty((n, self.k), dtype=torch.int32, device=words.device)
        with torch.cuda.device(words.device):
            timing.timed(f"cl_packed_network[{self.rows[0]}->{self.rows[-1]}]", lambda: _capi.call(
                "cl_packed_network", words.data_ptr(), row_bytes, n, self.tables.data_ptr(),
                self._rows_host, len(self.rows) - 1, self.k, counts.data_ptr(),
                _dl.stream_of(words)))
        return counts

    def _call_columns(self, x) -> torch.Tensor:
        """The wide-input path: the prefix layer by layer, the producer layer (or pair of
        layers) written column-major, then the fused tail on those columns."""
        if isinstance(x, PackBitsTensor):
            h = PackBitsTensor.from_packed(x.t, x.pad_len)   # the caller's object stays
        else:
            h = PackBitsTensor.from_packed(x)
        with torch.no_grad():
            for m in self.prefix:
                h = m(h)
            tabs = self._producer_tables()
        words, n = h.t, h.num_samples
        _dl._check(words, "x")
        if words.device != self.device:
            raise RuntimeError(f"x is on {words.device}, the network on {self.device}")
        in_rows = words.shape[0]
        expect = self._producer_rows()
        if in_rows != expect:
            raise RuntimeError(f"the layer before the fused tail gets {in_rows} rows, "
                               f"expects {expect}")
        if tabs[-1][0].numel() != self.rows[0]:
            raise RuntimeError(f"the layer before the fused tail has {tabs[-1][0].numel()} "
                               f"outputs, the tail reads {self.rows[0]}")
        row_bytes = words.shape[1] * words.element_size()
        if row_bytes % 4:
            raise RuntimeError("packed rows must be a multiple of 4 bytes")
        cols, in_words = row_bytes // 4, self.layout["in_words"]
        if self.circuit is not None and self._circuit_holds(tabs):
            if row_bytes * in_rows <= _ROWS_IN_CACHE:
                return self.circuit(words, cols, False, 0, n)
            with _dl.on_device_of(words):
                x = torch.empty((cols, in_rows), dtype=torch.int32, device=words.device)
                timing.timed(f"cl_packed_rows_to_columns[{in_rows}]", lambda: _capi.call(
                    "cl_packed_rows_to_columns", words.data_ptr(), x.data_ptr(), in_rows,
                    row_bytes, in_rows, _dl.stream_of(words)))
            return self.circuit(x, cols, True, in_rows, n)
        if self.tables is None:
            if torch.cuda.is_current_stream_capturing():
                return self._layer_by_layer(words, tabs, n)
            self._lay_out_rows()
        colmaj = torch.empty((cols, in_words), dtype=torch.int32, device=words.device)
        counts = torch.empty((n, self.k), dtype=torch.int32, device=words.device)
        stream = _dl.stream_of(words)
        ptrs = [t.data_ptr() for tab in tabs for t in tab]
        with torch.cuda.device(words.device):
            order = self.col_order.data_ptr()
            if len(tabs) == 2:
                mid = tabs[0][0].numel()
                timing.timed(f"cl_eval_packed_indexed_pair_columns[{in_rows}->{mid}->"
                             f"{self.rows[0]}]", lambda: _capi.call(
                    "cl_eval_packed_indexed_pair_columns", words.data_ptr(), *ptrs, order,
                    colmaj.data_ptr(), in_rows, mid, self.rows[0], row_bytes, in_words, stream))
            else:
                timing.timed(f"cl_eval_packed_indexed_columns[{in_rows}->{self.rows[0]}]",
                             lambda: _capi.call(
                    "cl_eval_packed_indexed_columns", words.data_ptr(), *ptrs, order,
                    colmaj.data_ptr(), in_rows, self.rows[0], row_bytes, in_words, stream))
            timing.timed(f"cl_packed_network_columns[{self.rows[0]}->{self.rows[-1]}]",
                         lambda: _capi.call(
                "cl_packed_network_columns", colmaj.data_ptr(), cols, in_words, n,
                self.tables.data_ptr(), self._rows_host, len(self.rows) - 1, self.k,
                counts.data_ptr(), stream))
        return counts

    def _front_pays(self, x) -> bool:
        words = x.t if isinstance(x, PackBitsTensor) else x
        rows = words.shape[0]
        known = self._front_from
        if known is None or known[0] != rows:
            known = self._front_from = (rows, tree_columns_from(self.front, rows))
        return words.shape[-1] * words.element_size() >= 4 * known[1]

    def _call_front(self, x):
        """The logic-tree blocks and the tail on columns: the packed rows turned to columns, all
        blocks on one column in LDS, then the fused tail.  None when the blocks' shape or taps
        (or the rows' width) ask for the layer-by-layer kernels."""
        words = x.t if isinstance(x, PackBitsTensor) else x
        _dl._check(words, "x")
        if words.dim() != 2 or words.device != self.device:
            return None
        rows, row_bytes = words.shape[0], words.shape[1] * words.element_size()
        blocks = self.front
        plan = tree_columns_layout(blocks, rows) if row_bytes and row_bytes % 8 == 0 else None
        if (plan is None or plan[1] != self.rows[0] or any(m.training for m in blocks)
                or not all(m._regular_taps() for m in blocks)
                or any(m.weights.device != self.device for m in blocks)
                or any(m._forward_hooks or m._forward_pre_hooks for m in blocks)):
            return None
        geo, _, table_words = plan
        n = x.num_samples if isinstance(x, PackBitsTensor) else row_bytes * 8
        cols, in_words = row_bytes // 4, self.front_layout["in_words"]
        dev, stream = words.device, _dl.stream_of(words)

        def ints(*shape):
            return torch.empty(shape, dtype=torch.int32, device=dev)

        with torch.no_grad(), _dl.on_device_of(words):
            gates = [m.weights.argmax(-1).to(torch.uint8).contiguous() for m in blocks]
            taps = [m.selection.to(torch.int32).contiguous() for m in blocks]
            ptrs = [(ctypes.c_void_p * len(blocks))(*[t.data_ptr() for t in ts])
                    for ts in (gates, taps)]
            colmaj, tables = ints(cols, rows), ints(table_words)
            timing.timed(f"cl_packed_rows_to_columns[{rows}]", lambda: _capi.call(
                "cl_packed_rows_to_columns", words.data_ptr(), colmaj.data_ptr(), rows,
                row_bytes, rows, stream))
            mid = ints(cols, in_words)
            timing.timed(f"cl_tree_columns[{rows}->{self.rows[0]}]", lambda: _capi.call(
                "cl_tree_columns", colmaj.data_ptr(), cols, rows, geo, len(blocks), *ptrs,
                tables.data_ptr(), mid.data_ptr(), in_words, stream))
            if self.circuit is not None:
                return self.circuit(mid, cols, True, in_words, n)
            counts = ints(n, self.k)
            timing.timed(f"cl_packed_network_columns[{self.rows[0]}->{self.rows[-1]}]",
                         lambda: _capi.call(
                "cl_packed_network_columns", mid.data_ptr(), cols, in_words, n,
                self.front_tables.data_ptr(), self._rows_host, len(self.rows) - 1, self.k,
                counts.data_ptr(), stream))
        return counts
