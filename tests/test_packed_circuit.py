"""The pruned circuit of a packed network (packed_circuit.fold / build): its tables, evaluated as
the kernel does, give the layers' class counts; on the GPU the kernel over several columns per
workgroup."""
import numpy as np
import pytest
import torch

from compactlogic_amd import packed_circuit as PC
from compactlogic_amd.packed_net import _Circuit

ALL = np.uint64(0xFFFFFFFFFFFFFFFF)


def random_layers(dims, seed, gates=range(16), strays=False):
    r = np.random.default_rng(seed)
    layers = []
    for i, o in dims:
        lo, hi = (-1, i + 1) if strays else (0, i)
        layers.append((r.integers(lo, hi, o), r.integers(lo, hi, o),
                       r.choice(np.array(list(gates)), o)))
    return layers


def words_of(gate, a, b):
    f = [np.where((gate >> s) & 1, ALL, np.uint64(0)) for s in (3, 2, 1, 0)]
    return (~a & ~b & f[0]) | (~a & b & f[1]) | (a & ~b & f[2]) | (a & b & f[3])


def reference_counts(layers, k, x):
    """A negative row reads 0; a row past the layer before makes the gate 0."""
    h = x
    for a, b, g in layers:
        rows = h.size
        h = np.append(h, np.uint64(0))
        bad = (a >= rows) | (b >= rows)
        av, bv = (h[np.where((v < 0) | (v >= rows), rows, v)] for v in (a, b))
        h = words_of(np.where(bad, 0, g), av, bv)
    bits = (h[:, None] >> np.arange(64, dtype=np.uint64)) & np.uint64(1)
    return bits.reshape(k, -1, 64).sum(1).T.astype(np.int64)


def table_counts(plan, k, x, rng):
    """The kernel's walk over the tables on one column of 64 samples; every step reads the words
    as they were when it began, and the next column's input is staged before the counts."""
    pairs, start, groups, inverted, in_pages, kk, pages = plan["shape"]
    assert kk == k
    lds = rng.integers(0, 2**63, 128 * pages).astype(np.uint64)   # a signal at its first word
    lds[:64] = 0
    rows = plan["in"][:64 * in_pages].astype(np.int64)
    at = 128 * (1 + np.arange(rows.size) // 64) + np.arange(rows.size) % 64
    rows, at = rows[rows != 0xFFFF], at[rows != 0xFFFF]
    lds[at] = x[rows]
    dst = np.stack([plan["dst"] & 0xFFFF, plan["dst"] >> 16], 2).reshape(16, -1)
    for b in range(pairs):
        if b == 0 or (start >> b) & 1:
            old = lds.copy()
        for q in (2 * b, 2 * b + 1):
            for w in range(16):
                page = int(dst[w, q])
                if page == 0xFFFF:
                    continue
                e = plan["ent"][q, 64 * w:64 * w + 64].astype(np.int64)
                o = plan["ops"][q // 8, 64 * w:64 * w + 64].astype(np.int64) >> (4 * (q % 8))
                gate = (o & 1) << 2 | (o & 2) | (o & 4) >> 2
                lds[page:page + 64] = words_of(gate, old[e & 0xFFFF], old[e >> 16])
    lds[at] = rng.integers(0, 2**63, rows.size).astype(np.uint64)
    out = np.tile(plan["ones"].astype(np.int64), (64, 1))
    if groups + inverted:
        cnt = plan["cnt"]
        at = np.stack([cnt & 0xFFFF, cnt >> 16], 4).reshape(groups + inverted, k, 64, 4)
        v = lds[at]
        v[groups:] = ~v[groups:]
        bits = (v[..., None] >> np.arange(64, dtype=np.uint64)) & np.uint64(1)
        out += bits.sum((0, 2, 3)).T.astype(np.int64)
    return out


CASES = [
    ([(40, 64), (64, 60)], 6, range(16), False),
    ([(17, 33), (33, 40)], 5, range(16), True),              # rows outside the layer before
    ([(12, 20)] + [(20, 20)] * 14 + [(20, 30)], 3, range(16), False),
    ([(6, 10)], 10, (3, 5, 10, 12), False),                  # outputs are inputs only
    ([(6, 10)], 2, (0, 15), False),                          # constants only
    ([(50, 700), (700, 640)], 1, (1, 6, 8, 9), False),       # one class, whole pages of a kind
    ([(300, 6000), (6000, 5000)], 20, range(16), False),
    ([(64, 11000), (11000, 12000)], 10, (1, 2, 4, 6, 7, 8, 9, 11, 13, 14), False),  # steps split
    ([(1500, 2000), (2000, 900)], 3, range(16), False),      # an input page per wave
    ([(9000, 12000), (12000, 3000)], 10, (1, 2, 4, 6, 7, 8, 9, 11, 13, 14), False),  # eight pages
    ([(6000, 4000), (4000, 3000)], 10, (1, 2, 4, 6, 7, 8, 9, 11, 13, 14), False),    # eight pages
    ([(3000, 3000), (3000, 3000)], 10, (1, 2, 4, 6, 7, 8, 9, 11, 13, 14), False),    # four pages
]


TWO = (1, 2, 4, 6, 7, 8, 9, 11, 13, 14)     # opcodes of both operands


def chain(first, width, layers):
    return [(first, width)] + [(width, width)] * (layers - 1)


# The kernel's variants: the gate slots and count planes it is compiled for, input pages per wave
# (16: two rounds of eight), and whether a step begins inside a block of four slots.
VARIANTS = [
    (chain(100, 2000, 19), 10, range(16), 40, 5, 1, True),
    (chain(100, 1100, 21), 10, TWO, 48, 5, 1, True),
    (chain(64, 3500, 10), 1, TWO, 40, 9, 1, False),
    ([(9200, 12000)] + chain(12000, 6000, 5), 2, TWO, 48, 9, 8, False),
    ([(1800, 3000), (3000, 2000)], 10, TWO, 32, 5, 2, False),
    ([(9400, 11000)], 1, TWO, 32, 9, 16, False),
    ([(9400, 11000)], 100, TWO, 32, 5, 16, False),
    (chain(8400, 4500, 8), 10, TWO, 40, 5, 8, False),
    (chain(600, 6500, 6), 50, TWO, 48, 5, 1, False),
]


@pytest.mark.parametrize("dims,k,gates,slots,planes,inputs,inside", VARIANTS)
def test_tables_of_every_kernel_variant(dims, k, gates, slots, planes, inputs, inside):
    rng = np.random.default_rng(k)
    layers = random_layers(dims, k, gates)
    plan = PC.build(PC.fold(layers, dims[0][0]), k)
    pairs, start, groups, inverted, in_pages = plan["shape"][:5]
    assert next(v for v in (32, 40, 48) if 2 * pairs <= v) == slots
    assert (5 if 4 * (groups + inverted) < 32 else 9) == planes
    assert next(v for v in (1, 2, 4, 8, 16) if in_pages <= 16 * v) == inputs
    assert any((start >> b) & 1 for b in range(1, pairs, 2)) == inside
    x = rng.integers(0, 2**63, dims[0][0]).astype(np.uint64)
    assert np.array_equal(table_counts(plan, k, x, rng), reference_counts(layers, k, x))


@pytest.mark.parametrize("dims,k,gates,strays", CASES)
def test_tables_give_the_layers_counts(dims, k, gates, strays):
    rng = np.random.default_rng(k)
    layers = random_layers(dims, k, gates, strays)
    plan = PC.build(PC.fold(layers, dims[0][0]), k)
    for _ in range(2):
        x = rng.integers(0, 2**63, dims[0][0]).astype(np.uint64)
        assert np.array_equal(table_counts(plan, k, x, rng), reference_counts(layers, k, x))


def test_what_does_not_fit_is_refused():
    lim = PC.limits()
    rows = 64 * lim["input_pages"]
    wide = random_layers([(rows, 64 * lim["pages"])], 1, (1, 6))
    assert PC.build(PC.fold(wide, rows), 1) is None                          # pages
    many = random_layers([(2 * rows, 16000)], 2, (1, 6))
    assert PC.build(PC.fold(many, 2 * rows), 1000) is None                   # input pages
    tall = random_layers([(64, 128 * lim["steps"])], 3, (3, 5))
    assert PC.build(PC.fold(tall, 64), 1) is None                            # entries of a class


def test_what_cannot_fit_is_not_placed(monkeypatch):
    """A circuit of more gates than slots, or that finds no page at any split, is refused without
    laying its signals out: the placement takes seconds over all the tries."""
    def placed(*args):
        raise AssertionError("a circuit that cannot fit was placed")

    monkeypatch.setattr(PC, "_Banks", placed)
    for dims in ([784] + [12000] * 6,             # 61000 gates, 49152 slots
                 [784, 16000, 16000],             # pages: only a schedule shows it
                 [30000, 20000, 20000]):          # more input pages than the kernel stages
        layers = random_layers(list(zip(dims[:-1], dims[1:])), 1, TWO)
        assert PC.build(PC.fold(layers, dims[0]), 10) is None


def test_where_a_circuit_pays():
    """Few gates saved and many classes, or one class of many rows, take the row tables without
    a placement; what `pays` allows is laid out."""
    def built(dims, k, gates, row_slots):
        layers = random_layers(list(zip(dims[:-1], dims[1:])), k, gates)
        return PC.build(PC.fold(layers, dims[0]), k, row_slots) is not None

    narrow = [784, 2000, 2000]                    # two slots per layer
    assert built(narrow, 10, TWO, 4) and not built(narrow, 200, TWO, 4)
    assert not built(narrow, 50, range(16), 4) and built(narrow, 50, range(16), None)
    wide = [784, 12000, 12000]
    assert built(wide, 2, range(16), 24) and not built(wide, 1, range(16), 24)


@pytest.mark.gpu
@pytest.mark.parametrize("dims,k,gates,strays",
                         CASES + [(*v[:3], False) for v in VARIANTS])
@pytest.mark.parametrize("n", [40000, 33])
def test_circuit_kernel(device, dims, k, gates, strays, n):
    """Several columns per workgroup (256 workgroups take 16384 samples at a time), row-major and
    column-major input."""
    rng = np.random.default_rng(k)
    layers = random_layers(dims, k, gates, strays)
    rows = dims[0][0]
    cols = -(-n // 32)
    x = rng.integers(0, 2**32, (rows, cols), dtype=np.uint64).astype(np.uint32)
    wide = np.zeros((rows, cols + cols % 2), dtype=np.uint32)
    wide[:, :cols] = x
    ref = np.concatenate([reference_counts(layers, k, c)
                          for c in wide.view(np.uint64).T])[:n]
    circuit = _Circuit.of(layers, rows, k, device)
    xt = torch.as_tensor(x.view(np.int32), device=device)
    assert np.array_equal(circuit(xt, cols, False, 0, n).cpu().numpy(), ref)
    pitch = rows + 3
    xc = torch.full((cols, pitch), -1, dtype=torch.int32, device=device)
    xc[:, :rows] = xt.t()
    assert np.array_equal(circuit(xc, cols, True, pitch, n).cpu().numpy(), ref)
