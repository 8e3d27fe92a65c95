"""A frozen network's tail as a pruned circuit on LDS pages: the tables of cl_packed_circuit
(csrc/packed_circuit.hip).

`fold` reduces the layers to the two-input gates that reach an output: constants and
pass-through gates are folded into their readers (inversions too), gates that nothing reads are
dropped.  The class counts are those of the network for every input.  This is the stage-1
pruning idea of the reference's compiler (compiler/prune.py:164-367) applied to the packed
evaluator's tables.

`build` schedules the gates in steps (a barrier between them; a gate's sources come from earlier
steps), places every signal in LDS and lays the tables out.  A page is 64 words, the gates of one
wave; it is reused after the last step that reads one of its signals, so signals that are last
read in the same step share pages.
"""
from __future__ import annotations

import ctypes
import heapq

import numpy as np

from . import _capi

_PAGE = 64
_WAVES = 16
_THREADS = 1024
_BATCH = 4          # slots per batch; a step begins with a batch
# smallest number of a step's gates with a death step of their own, in the order tried: fewer
# groups read LDS with fewer bank conflicts, more free pages earlier
_MIN_GROUPS = (1024, 192)


def limits() -> dict:
    v = [ctypes.c_int64(0) for _ in range(4)]
    _capi.call("cl_packed_circuit_limits", *[ctypes.byref(c) for c in v])
    return dict(zip(("words", "slots", "steps", "inputs"), (c.value for c in v)))


# truth tables as columns (00, 01, 10, 11) over (a, b); column orders of the foldings below
_NOT_A, _NOT_B = [2, 3, 0, 1], [1, 0, 3, 2]
_A0, _A1, _B0, _B1, _SAME = [0, 1, 0, 1], [2, 3, 2, 3], [0, 0, 2, 2], [1, 1, 3, 3], [0, 0, 3, 3]


def fold(layers: list, in_rows: int) -> dict:
    """layers: (a, b, opcode) int arrays per layer, a and b rows of the layer before (a negative
    row is 0; a row past the layer before makes the gate 0).  Signals are numbered inputs first,
    then the two-input gates in layer order; a gate that is 1 for a = b = 0 is kept inverted, and
    its readers take that up.  Returns a, b, bits (the gate's values for ab = 01, 10, 11 in bits
    0, 1, 2), layer of the gates, and the outputs' signal (-1: constant), inverted, constant,
    with live [signals] whether an output depends on the signal."""
    sig = np.arange(in_rows, dtype=np.int64)
    inv = np.zeros(in_rows, dtype=bool)
    const = np.full(in_rows, -1, dtype=np.int64)
    ga, gb, gt, gl = [], [], [], []
    nxt = in_rows
    for l, (a, b, g) in enumerate(layers):
        rows = sig.size
        past = (a >= rows) | (b >= rows)
        # row `rows` of the extended arrays is the constant 0
        sig, inv, const = np.append(sig, -1), np.append(inv, False), np.append(const, 0)
        a, b = np.where((a < 0) | past, rows, a), np.where((b < 0) | past, rows, b)
        g = np.where(past, 0, g)
        t = np.stack([(g >> s) & 1 for s in (3, 2, 1, 0)], 1)
        for col, cond in ((_NOT_A, inv[a]), (_NOT_B, inv[b]), (_A0, const[a] == 0),
                          (_A1, const[a] == 1), (_B0, const[b] == 0), (_B1, const[b] == 1),
                          (_SAME, (sig[a] == sig[b]) & (const[a] < 0) & (const[b] < 0))):
            t = np.where(cond[:, None], t[:, col], t)
        on_a = (t[:, 0] != t[:, 2]) | (t[:, 1] != t[:, 3])
        on_b = (t[:, 0] != t[:, 1]) | (t[:, 2] != t[:, 3])
        sa, sb = sig[a], sig[b]
        two = on_a & on_b
        n = int(two.sum())
        sig = np.where(on_a, sa, np.where(on_b, sb, -1))
        sig[two] = nxt + np.arange(n)
        inv = (t[:, 0] == 1) & (on_a | on_b)
        const = np.where(on_a | on_b, -1, t[:, 0])
        f = t[two] ^ t[two][:, :1]
        ga.append(sa[two]), gb.append(sb[two])
        gt.append(f[:, 1] | f[:, 2] << 1 | f[:, 3] << 2)
        gl.append(np.full(n, l, dtype=np.int64))
        nxt += n
    a, b, t, layer = (np.concatenate(v) for v in (ga, gb, gt, gl))
    live = np.zeros(nxt, dtype=bool)
    live[sig[const < 0]] = True
    for l in range(len(layers) - 1, -1, -1):
        q = np.nonzero((layer == l) & live[in_rows:])[0]
        live[a[q]] = live[b[q]] = True
    return {"in_rows": in_rows, "a": a, "b": b, "bits": t, "layer": layer, "out": sig,
            "out_inv": inv, "out_const": const, "live": live}


def _groups(death: np.ndarray, smallest: int) -> list:
    """Index groups of equal death step, earliest first; groups below `smallest` join the next
    later one."""
    out, rest = [], np.zeros(0, dtype=np.int64)
    for d in np.unique(death):
        rest = np.concatenate((rest, np.nonzero(death == d)[0]))
        if rest.size >= smallest:
            out.append(rest)
            rest = np.zeros(0, dtype=np.int64)
    if rest.size:
        out.append(rest)
    return out


_I32, _I64 = ctypes.POINTER(ctypes.c_int32), ctypes.POINTER(ctypes.c_int64)


def _host(a, dtype):
    a = np.ascontiguousarray(a, dtype=dtype)
    return a, a.ctypes.data_as(_I32 if dtype == np.int32 else _I64)


class _Banks:
    """Bank placement of signals.  The signals that one group of gates reads are spread evenly
    over the banks when they are placed, the gates' operands are ordered so that either operand's
    reads are, and the gates are put into half-waves that read every bank once."""

    def __init__(self, reader: np.ndarray, source: np.ndarray, signals: int, groups: int):
        order = np.argsort(source, kind="stable")
        self.reader = reader[order]
        self.ptr = np.searchsorted(source[order], np.arange(signals + 1))
        self.load = np.zeros((groups, 32), dtype=np.int64)

    def slots(self, signals: np.ndarray) -> np.ndarray:
        """signals (in blocks of 32) in the order of their words."""
        n = signals.size
        count = self.ptr[signals + 1] - self.ptr[signals]
        ptr = np.concatenate(([0], np.cumsum(count)))
        at = np.repeat(self.ptr[signals] - ptr[:-1], count) + np.arange(ptr[-1])
        (ptr, p), (grp, g), (slot, s) = (_host(ptr, np.int64), _host(self.reader[at], np.int32),
                                         _host(np.zeros(n), np.int32))
        _capi.call("cl_packed_bank_slots", p, g, n, self.load.shape[0],
                   self.load.ctypes.data_as(_I64), s)
        out = np.empty_like(signals)
        out[np.arange(n) // 32 * 32 + slot] = signals
        return out

    @staticmethod
    def orient(wa: np.ndarray, wb: np.ndarray) -> np.ndarray:
        """Gates that read operands at words wa, wb: those to swap."""
        (ka, a), (kb, b), (swap, s) = (_host(wa % 32, np.int32), _host(wb % 32, np.int32),
                                       _host(np.zeros(wa.size), np.int32))
        _capi.call("cl_packed_bank_orient", a, b, wa.size, s)
        return swap.astype(bool)


def _by_bank(w: np.ndarray) -> np.ndarray:
    """w in an order that takes every LDS bank in turn."""
    by = np.argsort(w % 32, kind="stable")
    banks = (w % 32)[by]
    rank = np.empty(w.size, dtype=np.int64)
    rank[by] = np.arange(w.size) - np.searchsorted(banks, banks)
    return w[np.lexsort((w % 32, rank))]


def build(c: dict, k: int, splits=(1, 2, 3, 4)) -> dict | None:
    """Tables for fold's result c with k classes, or None when the circuit does not fit.  A level
    split into more steps frees its sources' pages earlier and costs barriers: the first split
    that fits is taken."""
    lim = limits()
    for split in splits:
        for smallest in _MIN_GROUPS:
            plan = _build(c, k, split, smallest, lim)
            if plan is not None:
                return plan
    return None


def _build(c: dict, k: int, split: int, smallest: int, lim: dict) -> dict | None:
    from .packed_net import bank_aware_positions

    n_in, a, b, bits = c["in_rows"], c["a"].copy(), c["b"].copy(), c["bits"].copy()
    live, layer = c["live"], c["layer"]
    steps = []
    for l in np.unique(layer):
        q = np.nonzero((layer == l) & live[n_in:])[0]
        if q.size:
            parts = min(split, max(1, q.size // (_PAGE * _WAVES)))
            steps += np.array_split(q, parts)
    end = len(steps)
    death = np.full(live.size, -1, dtype=np.int64)
    for s, q in enumerate(steps):
        death[a[q]] = death[b[q]] = s
    is_out = c["out_const"] < 0
    death[c["out"][is_out]] = end
    steps = [[q[g] for g in _groups(death[n_in + q], smallest)] for q in steps]
    groups = [g for step in steps for g in step]
    gates = np.concatenate(groups) if groups else np.zeros(0, dtype=np.int64)
    gid = np.repeat(np.arange(len(groups)), [g.size for g in groups])
    banks = _Banks(np.concatenate((gid, gid)), np.concatenate((a[gates], b[gates])), live.size,
                   len(groups))

    max_pages = lim["words"] // _PAGE
    free = list(range(1, max_pages))               # page 0: zeros
    word = np.full(live.size, -1, dtype=np.int64)
    dying = [[] for _ in range(end + 1)]
    peak = 1

    ins = np.nonzero(live[:n_in])[0]
    if ins.size > lim["inputs"]:
        return None
    in_pages = 0
    for grp in _groups(death[ins], smallest):
        ids = banks.slots(ins[grp])
        for p0 in range(0, ids.size, _PAGE):
            if not free:
                return None
            page = heapq.heappop(free)
            part = ids[p0:p0 + _PAGE]
            word[part] = page * _PAGE + np.arange(part.size)
            dying[int(death[part].max())].append(page)
            in_pages = max(in_pages, page + 1)
    peak = max(peak, in_pages)

    slots, start, ent, dst = 0, 0, [], []
    for s, step in enumerate(steps):
        pages = []
        for g in step:
            swap = banks.orient(word[a[g]], word[b[g]])
            a[g], b[g] = np.where(swap, b[g], a[g]), np.where(swap, a[g], b[g])
            bits[g] = np.where(swap, bits[g] & 4 | bits[g] >> 1 & 1 | bits[g] << 1 & 2, bits[g])
            pos = bank_aware_positions(word[a[g]], word[b[g]], g.size)
            order = np.empty_like(g)
            order[pos] = g
            order = banks.slots(n_in + order) - n_in
            for p0 in range(0, order.size, _PAGE):
                part = order[p0:p0 + _PAGE]
                last = int(death[n_in + part].max())
                # gates the counts read stay off the input pages, which the next column's
                # input is staged to while the counts run
                skip = []
                while free and last == end and free[0] < in_pages:
                    skip.append(heapq.heappop(free))
                if not free:
                    return None
                page = heapq.heappop(free)
                for v in skip:
                    heapq.heappush(free, v)
                peak = max(peak, page + 1)
                word[n_in + part] = page * _PAGE + np.arange(part.size)
                dying[last].append(page)
                pages.append((page, part))
        need = -(-len(pages) // _WAVES)
        need = -(-need // _BATCH) * _BATCH
        if slots + need > lim["slots"]:
            return None
        start |= 1 << (slots // _BATCH)
        e = np.zeros((need, _THREADS), dtype=np.uint32)
        d = np.full((_WAVES, need), 0xFFFF, dtype=np.uint32)
        for i, (page, part) in enumerate(pages):
            w, j = i % _WAVES, i // _WAVES
            t = bits[part]
            e[j, w * _PAGE + np.arange(part.size)] = \
                4 * word[a[part]] | 4 * word[b[part]] << 16 | t & 3 | (t & 4) << 14
            d[w, j] = page * _PAGE
        slots += need
        ent.append(e), dst.append(d)
        for page in dying[s]:
            heapq.heappush(free, page)

    pad = lim["slots"] - slots
    dst_all = np.concatenate(dst + [np.full((_WAVES, pad), 0xFFFF, dtype=np.uint32)], 1)

    # outputs: per class the words counted as they are and those counted inverted, each padded
    # with the zero page to whole groups of four entries per lane
    out, inv, const = c["out"], c["out_inv"], c["out_const"]
    gs = out.size // k
    ones = np.array([int((const[i * gs:(i + 1) * gs] == 1).sum()) for i in range(k)])
    groups, cnt = [], []
    for flip in (False, True):
        lists = []
        for cls in range(k):
            r = np.arange(cls * gs, (cls + 1) * gs)
            lists.append(_by_bank(word[out[r[(const[r] < 0) & (inv[r] == flip)]]]))
        n = max(-(-v.size // (4 * _PAGE)) for v in lists)
        tab = np.tile(np.arange(_PAGE, dtype=np.int64), (k, 4 * n, 1))    # the zero page
        for cls, v in enumerate(lists):
            tab[cls].reshape(-1)[:v.size] = v
            if flip:
                ones[cls] -= 4 * n * _PAGE - v.size
        groups.append(n)
        # [group][class][lane][2]: four byte addresses of 16 bits
        t = 4 * tab.reshape(k, n, 2, 2, _PAGE)
        cnt.append((t[:, :, :, 0] | (t[:, :, :, 1] << 16)).transpose(1, 0, 3, 2))
    if 4 * sum(groups) > lim["steps"]:
        return None
    cnt = np.ascontiguousarray(np.concatenate(cnt)).astype(np.uint32)
    return {
        "shape": (slots // _BATCH, start, groups[0], groups[1], int(ins.size), k, peak * _PAGE,
                  int((out[is_out] < n_in).any())),
        "ent": np.concatenate(ent) if ent else np.zeros((1, _THREADS), dtype=np.uint32),
        "dst": (dst_all[:, 0::2] | (dst_all[:, 1::2] << 16)).astype(np.uint32),
        "in": (ins | (word[ins] << 16)).astype(np.uint32) if ins.size else
        np.zeros(1, dtype=np.uint32),
        "cnt": cnt if cnt.size else np.zeros(1, dtype=np.uint32),
        "ones": ones.astype(np.int32),
        "gates": int(gates.size), "levels": end,
    }
