"""Whole-network packed inference (PackedNetwork): bit-exact against the C oracle and the
layer-by-layer packed path."""
import numpy as np
import pytest
import torch

import compactlogic_amd as cl
from compactlogic_amd import configs
from oracle import packed as P

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def columns_at_every_size(request, monkeypatch):
    """The column pass of logic-tree blocks at any size and shape, for the tests of its kernels."""
    if "tree_front" in request.node.name:
        from compactlogic_amd import packed_net
        monkeypatch.setattr(packed_net, "tree_columns_from", lambda blocks, rows: 0)


def np_(t):
    return t.detach().cpu().numpy()


def frozen_net(dims, k, g_n, seed, device):
    torch.manual_seed(seed)
    layers = [cl.LogicLayer(i, o, num_gates=g_n) for i, o in dims]
    g = torch.Generator().manual_seed(seed)
    for m in layers:
        with torch.no_grad():
            m.gate_sequence.copy_(torch.randint(0, 16, m.gate_sequence.shape, generator=g).to(torch.uint8))
        m.freeze()
    model = torch.nn.Sequential(*layers, cl.GroupSum(k, 1.0)).to(device)
    model.eval()
    return model


def oracle_counts(model, words_np, n):
    layers = [P.resolve_slots(np_(m.indices), np_(m.gate_sequence), np_(m.w))
              for m in model if isinstance(m, cl.LogicLayer)]
    pad = words_np.shape[1] * 64 - n
    return P.network_counts(words_np, layers, model[-1].k, pad)


@pytest.mark.parametrize("dims,k,g_n,n", [
    ([(40, 64), (64, 60)], 6, 4, 64),
    ([(100, 300), (300, 300), (300, 200)], 10, 16, 1000),
    ([(17, 33), (33, 40)], 5, 2, 96),
    ([(64, 2000), (2000, 1000)], 8, 16, 4096),
    ([(12, 20)] + [(20, 20)] * 14 + [(20, 30)], 3, 8, 130),
    ([(64, 17000), (17000, 8500)], 10, 4, 200),     # wider than the register-table variant
    ([(3000, 5000), (5000, 2600)], 4, 16, 700),     # > 1024 input rows: 4 per thread
    ([(64, 15000), (15000, 16000)], 2, 4, 300),     # 16 gates per thread, 8000-row classes
    ([(50, 400), (400, 340)], 20, 8, 150),          # more classes than waves
])
def test_packed_network_matches_oracle_and_layerwise(device, dims, k, g_n, n):
    model = frozen_net(dims, k, g_n, sum(d[1] for d in dims), device)
    rng = np.random.default_rng(n)
    bits = rng.integers(0, 2, (n, dims[0][0])).astype(bool)
    x = cl.PackBitsTensor(torch.as_tensor(bits, device=device), 64)
    net = cl.PackedNetwork(model)
    counts = net(x)
    assert counts.shape == (n, k) and counts.dtype == torch.int32
    ref = oracle_counts(model, np_(x.t).view(np.uint64), n)
    assert np.array_equal(np_(counts), ref)
    layerwise = model(cl.PackBitsTensor.from_packed(x.t.clone(), x.pad_len))
    assert torch.equal(counts, layerwise)


def conv_oracle_counts(model, words_np, n):
    """The C oracle through a network of ConvLayers, Flatten and LogicLayers."""
    layers = []
    for m in model:
        if isinstance(m, cl.ConvLayer):
            layers.append(P.resolve_conv_slots(np_(m.offsets_ch), np_(m.offsets_h),
                                               np_(m.offsets_w), np_(m.gate_sequence), np_(m.w),
                                               m.in_shape, m.stride, m.out_shape[1:]))
        elif isinstance(m, cl.LogicLayer):
            layers.append(P.resolve_slots(np_(m.indices), np_(m.gate_sequence), np_(m.w)))
    pad = words_np.shape[1] * 64 - n
    return P.network_counts(words_np, layers, model[-1].k, pad)


def test_packed_network_cfg5_fuses_the_wide_tail(device):
    """cfg5: conv1 and conv2 composed into one launch that writes conv2's rows column-major
    (conv1's rows computed where conv2 reads them), then 25088 -> 16000 -> 16000 and the class
    counts in one launch (two first-layer slots held over the input column); equal to the C
    oracle and to the whole network layer by layer."""
    cfg = configs.CONV_CONFIGS["cfg5"]
    model = configs.conv_network(cfg, device=device)
    configs.freeze_argmax(model)
    feats = int(np.prod(cfg.in_shape))
    xw = configs.packed_input_words(feats, 64, device=device)            # 2^12 samples
    net = cl.PackedNetwork(model)
    assert net.producer == (model[0], model[1]) and net.prefix == []
    assert net.rows == [25088, 16000, 16000] and net.layout["split"] == 14336
    x = cl.PackBitsTensor.from_packed(xw)
    counts = net(x)
    assert x.t is xw                                                     # input untouched
    ref = conv_oracle_counts(model, np_(xw).view(np.uint64), 1 << 12)
    assert np.array_equal(np_(counts), ref)
    assert torch.equal(counts, model(cl.PackBitsTensor.from_packed(xw.clone())))


def small_conv_net(device, in_shape, c_out, widths, k, seed, convs=1, stride=1):
    torch.manual_seed(seed)
    conv, shape = [], in_shape
    for i in range(convs):
        conv.append(cl.ConvLayer(shape, padding=1, c_out=c_out, ks=3, stride=stride,
                                 num_chn=1, num_gates=4))
        shape = conv[-1].out_shape
    g = torch.Generator().manual_seed(seed)
    dims = [int(np.prod(shape))] + list(widths)
    dense = [cl.LogicLayer(i, o, num_gates=4) for i, o in zip(dims[:-1], dims[1:])]
    for m in conv + dense:
        with torch.no_grad():
            m.weights.copy_(torch.randn(m.weights.shape, generator=g))
            m.gate_sequence.copy_(torch.randint(0, 16, m.gate_sequence.shape,
                                                generator=g).to(torch.uint8))
    model = torch.nn.Sequential(*conv, torch.nn.Flatten(), *dense,
                                cl.GroupSum(k, 1.0)).to(device)
    configs.freeze_argmax(model)
    return model


@pytest.mark.parametrize("in_shape,c_out,widths,k,n,bits", [
    ((4, 16, 16), 32, [4200, 2100], 10, 1000, 64),     # 8 slots, second layer over the input
    ((2, 12, 12), 40, [12000, 10000], 10, 333, 64),    # 16 slots, nothing held
    ((5, 15, 15), 40, [12000, 10000], 20, 100, 32),    # 9000 rows: held slots; odd words
    ((3, 16, 16), 24, [5000, 4000, 2100], 3, 4096, 64),  # three layers
])
def test_packed_network_wide_tail_matches_oracle(device, in_shape, c_out, widths, k, n, bits):
    model = small_conv_net(device, in_shape, c_out, widths, k, seed=n)
    rng = np.random.default_rng(n)
    feats = int(np.prod(in_shape))
    x = cl.PackBitsTensor(torch.as_tensor(rng.integers(0, 2, (n, feats)).astype(bool),
                                          device=device), bits)
    net = cl.PackedNetwork(model)
    assert net.producer == (model[0],) and net.layout is not None
    counts = net(x)
    assert counts.shape == (n, k)
    words = np_(x.t)
    if words.dtype != np.int64:                  # 32-bit words: pad to whole 64-bit words
        words = np.concatenate([words, np.zeros((words.shape[0], words.shape[1] % 2),
                                                words.dtype)], 1)
    ref = conv_oracle_counts(model, np.ascontiguousarray(words).view(np.uint64), n)
    assert np.array_equal(np_(counts), ref)
    layerwise = model(cl.PackBitsTensor.from_packed(x.t.clone(), x.pad_len))
    assert torch.equal(counts, layerwise)


def test_packed_network_wide_tail_after_a_dense_producer(device):
    """A dense LogicLayer feeds the tail through a Flatten: it writes the columns."""
    model = frozen_net([(64, 6000), (6000, 3000), (3000, 2000)], 10, 8, 11, device)
    model = torch.nn.Sequential(model[0], torch.nn.Flatten(), model[1], model[2], model[3])
    net = cl.PackedNetwork(model)
    assert net.producer == (model[0],) and net.prefix == [] and net.rows == [6000, 3000, 2000]
    rng = np.random.default_rng(3)
    x = cl.PackBitsTensor(torch.as_tensor(rng.integers(0, 2, (777, 64)).astype(bool),
                                          device=device), 64)
    counts = net(x)
    ref = oracle_counts(model, np_(x.t).view(np.uint64), 777)
    assert np.array_equal(np_(counts), ref)


@pytest.mark.parametrize("in_shape,c_out,convs,stride,widths,k,n", [
    ((3, 16, 16), 32, 2, 1, [4200, 2100], 10, 1000),   # conv, conv composed, 8192 rows
    ((4, 16, 16), 24, 3, 1, [3100, 1550], 5, 333),     # conv layer by layer, then a pair
])
def test_packed_network_composes_two_convs(device, in_shape, c_out, convs, stride, widths, k,
                                           n):
    model = small_conv_net(device, in_shape, c_out, widths, k, seed=n, convs=convs,
                           stride=stride)
    net = cl.PackedNetwork(model)
    assert net.producer == (model[convs - 2], model[convs - 1])
    assert net.prefix == list(model)[:convs - 2]
    rng = np.random.default_rng(n)
    feats = int(np.prod(in_shape))
    x = cl.PackBitsTensor(torch.as_tensor(rng.integers(0, 2, (n, feats)).astype(bool),
                                          device=device), 64)
    counts = net(x)
    ref = conv_oracle_counts(model, np_(x.t).view(np.uint64), n)
    assert np.array_equal(np_(counts), ref)
    assert torch.equal(counts, model(cl.PackBitsTensor.from_packed(x.t.clone(), x.pad_len)))


@pytest.mark.parametrize("mid,out_dim,out_words,words", [
    (500, 1000, 1024, 130), (300, 64, 64, 64), (40, 70, 128, 3)])
def test_eval_packed_indexed_pair_columns_is_two_layers(device, mid, out_dim, out_words, words):
    """The composed pair equals layer 1 by cl_eval_packed_indexed, then layer 2 written
    column-major; negative and out-of-range indices in both layers."""
    from compactlogic_amd import _capi
    from compactlogic_amd import difflogic_hip as _dl
    rng = np.random.default_rng(mid + out_dim)
    in_dim = 200
    xw = torch.as_tensor(rng.integers(-2**31, 2**31, (in_dim, words)), dtype=torch.int32,
                         device=device)

    def tables(n_in, n_out):
        ia = rng.integers(-1, n_in, n_out).astype(np.int32)
        ib = rng.integers(-1, n_in, n_out).astype(np.int32)
        ib[::13] = n_in                                   # out of range: a zero row
        g = rng.integers(0, 16, n_out).astype(np.uint8)
        return [torch.as_tensor(t, device=device) for t in (ia, ib, g)]

    t1, t2 = tables(in_dim, mid), tables(mid, out_dim)
    row_bytes = words * 4
    s = _dl.stream_of(xw)
    h = torch.empty((mid, words), dtype=torch.int32, device=device)
    _capi.call("cl_eval_packed_indexed", xw.data_ptr(), *[t.data_ptr() for t in t1], None,
               h.data_ptr(), in_dim, mid, row_bytes, s)
    ref = torch.full((words, out_words), 5, dtype=torch.int32, device=device)
    order = torch.as_tensor(rng.permutation(out_dim).astype(np.int32), device=device)
    _capi.call("cl_eval_packed_indexed_columns", h.data_ptr(), *[t.data_ptr() for t in t2],
               order.data_ptr(), ref.data_ptr(), mid, out_dim, row_bytes, out_words, s)
    out = torch.full((words, out_words), 7, dtype=torch.int32, device=device)
    _capi.call("cl_eval_packed_indexed_pair_columns", xw.data_ptr(),
               *[t.data_ptr() for t in t1 + t2], order.data_ptr(), out.data_ptr(), in_dim, mid,
               out_dim, row_bytes, out_words, s)
    torch.cuda.synchronize()
    assert torch.equal(out, ref)
    assert int(out[:, out_dim:].abs().sum()) == 0


@pytest.mark.parametrize("out_dim,out_words,words,bits", [
    (1000, 1024, 130, 32), (4096, 4096, 256, 32), (70, 128, 3, 32), (25, 64, 2, 64)])
def test_eval_packed_indexed_columns_is_the_transposed_layer(device, out_dim, out_words, words,
                                                             bits):
    """cl_eval_packed_indexed_columns equals cl_eval_packed_indexed transposed to 32-bit words,
    with zero rows past out_dim; negative and out-of-range indices as there."""
    from compactlogic_amd import _capi
    from compactlogic_amd import difflogic_hip as _dl
    rng = np.random.default_rng(out_dim)
    in_dim = 300
    xw = torch.as_tensor(rng.integers(-2**31, 2**31, (in_dim, words * bits // 32)),
                         dtype=torch.int32, device=device)
    ia = rng.integers(-1, in_dim, out_dim).astype(np.int32)
    ib = rng.integers(-1, in_dim, out_dim).astype(np.int32)
    ia[::17] = in_dim                                   # out of range: a zero row
    ia_t, ib_t = torch.as_tensor(ia, device=device), torch.as_tensor(ib, device=device)
    gate = torch.as_tensor(rng.integers(0, 16, out_dim).astype(np.uint8), device=device)
    row_bytes = xw.shape[1] * 4
    ref = torch.empty((out_dim, xw.shape[1]), dtype=torch.int32, device=device)
    _capi.call("cl_eval_packed_indexed", xw.data_ptr(), ia_t.data_ptr(), ib_t.data_ptr(),
               gate.data_ptr(), None, ref.data_ptr(), in_dim, out_dim, row_bytes,
               _dl.stream_of(xw))
    out = torch.full((xw.shape[1], out_words), 7, dtype=torch.int32, device=device)
    _capi.call("cl_eval_packed_indexed_columns", xw.data_ptr(), ia_t.data_ptr(),
               ib_t.data_ptr(), gate.data_ptr(), None, out.data_ptr(), in_dim, out_dim,
               row_bytes, out_words, _dl.stream_of(xw))
    torch.cuda.synchronize()
    assert torch.equal(out[:, :out_dim], ref.T)
    assert int(out[:, out_dim:].abs().sum()) == 0
    # with a row order: position p holds row order[p]
    order = torch.as_tensor(rng.permutation(out_dim).astype(np.int32), device=device)
    _capi.call("cl_eval_packed_indexed_columns", xw.data_ptr(), ia_t.data_ptr(),
               ib_t.data_ptr(), gate.data_ptr(), order.data_ptr(), out.data_ptr(), in_dim,
               out_dim, row_bytes, out_words, _dl.stream_of(xw))
    torch.cuda.synchronize()
    assert torch.equal(out[:, :out_dim], ref.T[:, order.long()])
    assert int(out[:, out_dim:].abs().sum()) == 0


def test_packed_network_cfg3_tree_fuses_the_dense_tail(device):
    """cfg3_tree: two ConvLogicLayer blocks layer by layer, then 2048 -> 16000 -> 16000 and
    the class counts in one launch; equal to the whole network layer by layer."""
    cfg = configs.TREE_CONFIGS["cfg3_tree"]
    model = configs.tree_network(cfg, device=device)
    configs.freeze_argmax(model)
    feats = int(np.prod(cfg.in_shape))
    xw = configs.packed_input_words(feats, 64, device=device)            # 2^12 samples
    net = cl.PackedNetwork(model)
    assert len(net.prefix) == 3 and net.rows == [2048, 16000, 16000]
    counts = net(cl.PackBitsTensor.from_packed(xw))
    layerwise = model(cl.PackBitsTensor.from_packed(xw.clone()))
    assert torch.equal(counts, layerwise)
    # the fused tail alone against the C oracle, on the blocks' packed output
    with torch.no_grad():
        h = cl.PackBitsTensor.from_packed(xw.clone())
        for m in net.prefix:
            h = m(h)
    dense = torch.nn.Sequential(*list(model)[3:])
    hw = np_(h.t).view(np.uint64)
    ref = oracle_counts(dense, hw, 1 << 12)
    assert np.array_equal(np_(counts), ref)


def test_packed_network_cfg4_slice(device):
    cfg = configs.CONFIGS["cfg2"]
    model = configs.dense_network(cfg, device=device)
    configs.freeze_uniform_gates(model)
    xw = configs.packed_input_words(cfg.in_dim, 1024, device=device)      # 2^16 samples
    counts = cl.PackedNetwork(model)(cl.PackBitsTensor.from_packed(xw))
    ref = oracle_counts(model, np_(xw).view(np.uint64), 1 << 16)
    assert np.array_equal(np_(counts), ref)


def test_packed_network_word_widths_and_errors(device):
    model = frozen_net([(30, 40), (40, 20)], 4, 4, 1, device)
    rng = np.random.default_rng(0)
    bits = rng.integers(0, 2, (200, 30)).astype(bool)
    ref = None
    for bc in (32, 64):
        x = cl.PackBitsTensor(torch.as_tensor(bits, device=device), bc)
        c = cl.PackedNetwork(model)(x)
        ref = c if ref is None else ref
        assert torch.equal(c, ref)
    bad = torch.nn.Sequential(*list(model)[:-1], cl.GroupSum(3, 1.0))
    with pytest.raises(ValueError):
        cl.PackedNetwork(bad)                                           # 20 % 3 != 0
    wide = frozen_net([(30, 30000)], 10, 2, 2, device)
    net = cl.PackedNetwork(wide)                                        # too wide for LDS
    assert net.rows is None
    x = cl.PackBitsTensor(torch.as_tensor(bits, device=device), 64)
    assert torch.equal(net(x), wide(cl.PackBitsTensor.from_packed(x.t.clone(), x.pad_len)))
    with pytest.raises(RuntimeError):
        cl.PackedNetwork(model)(torch.zeros((31, 4), dtype=torch.int64, device=device))


def test_bank_aware_layout_gives_the_same_counts(device):
    """The LDS layout of the hidden layers changes where rows live, never the counts."""
    dims = [(300, 2000), (2000, 3000), (3000, 1500)]
    model = frozen_net(dims, 10, 16, 5, device)
    n = 2048
    rng = np.random.default_rng(5)
    bits = rng.integers(0, 2, (n, 300)).astype(bool)
    x = cl.PackBitsTensor(torch.as_tensor(bits, device=device), 64)
    a = cl.PackedNetwork(model)(x)
    b = cl.PackedNetwork(model, bank_aware=False)(x)
    assert torch.equal(a, b)
    assert np.array_equal(np_(a), oracle_counts(model, np_(x.t).view(np.uint64), n))


def tree_net(blocks, dense, k, seed, device):
    torch.manual_seed(seed)
    mods = [cl.ConvLogicLayer(ci, co, stride=s, padding=p, kernel=ks, complete=True, num_chn=0)
            for ci, co, s, p, ks in blocks]
    model = torch.nn.Sequential(*mods, torch.nn.Flatten(),
                                *[cl.LogicLayer(i, o) for i, o in dense], cl.GroupSum(k, 1.0))
    model = model.to(device)
    configs.freeze_argmax(model)
    return model


@pytest.mark.parametrize("side,blocks,dense,n", [
    # 8 x 8 pooled positions (a wave per channel), then 4 per channel (a lane per position)
    (32, [(3, 40, 2, 1, 3), (40, 32, 2, 1, 3)], [(128, 300), (300, 200)], 1000),
    (32, [(9, 16, 2, 1, 3)], [(1024, 600)], 64),                   # one block
    (16, [(2, 17, 1, 1, 3)], [(1088, 1000), (1000, 990)], 333),    # stride 1: dy = pitch, 64 positions
    (64, [(1, 5, 2, 2, 5)], [(1280, 700)], 130),                   # 256 positions, kernel 5, pad 2
    (12, [(3, 10, 1, 1, 3), (10, 12, 1, 1, 3)], [(108, 200)], 77), # 36 positions, 9 positions
    (33, [(2, 9, 2, 0, 2)], [(576, 500)], 50),                     # odd side, even kernel, no halo
    (16, [(2, 6, 1, 1, 3), (6, 7, 1, 1, 3), (7, 8, 1, 1, 3)], [(32, 100)], 200),  # three blocks
])
def test_tree_front_on_columns(device, side, blocks, dense, n):
    """PackedNetwork runs complete logic-tree blocks on columns (cl_tree_columns): counts equal to
    the layer-by-layer kernels', which the oracle pins, at word counts off the column tiles."""
    from compactlogic_amd import timing
    model = tree_net(blocks, dense, 10, n, device)
    bits = torch.rand((n, blocks[0][0] * side * side), device=device) < 0.5
    x = cl.PackBitsTensor(bits, 64)
    net = cl.PackedNetwork(model)
    with timing.record() as rec:
        counts = net(x)
    assert any(c.startswith("cl_tree_columns") for c in rec.summary())
    ref = model(cl.PackBitsTensor.from_packed(x.t.clone(), x.pad_len))
    assert torch.equal(counts, ref)


def test_tree_front_every_gate_and_bad_channel(device):
    """cl_tree_columns against cl_tree_conv_eval_packed on one block with random gates for a wave
    per channel and a lane per position, every opcode at every node (all pairs over the
    channels), and channels whose taps name a channel past the input."""
    import ctypes
    from compactlogic_amd import _capi
    from compactlogic_amd import treelogic as TL
    rng = np.random.default_rng(5)
    for side, cin, cout, stride in ((32, 2, 700, 2), (8, 3, 700, 2)):
        gates = torch.as_tensor(rng.integers(0, 16, (cout, 7)).astype(np.uint8), device=device)
        sel = (rng.integers(0, cin, (cout, 8)) << 16) | (rng.integers(0, 3, (cout, 8)) << 8) \
            | rng.integers(0, 3, (cout, 8))
        sel[::97, 3] = cin << 16
        sel = torch.as_tensor(sel.astype(np.int32), device=device)
        words = 5
        xw = torch.as_tensor(rng.integers(-2**31, 2**31, (cin * side * side, 2 * words)),
                             dtype=torch.int32, device=device).view(torch.int64)
        ref = TL.tree_conv_eval_packed(xw, gates, sel, (cin, side, side), stride, 1, 3, True)
        geo = (ctypes.c_int64 * 10)(cin, side, side, cout, stride, stride, 1, 1, 3, 3)
        v = [ctypes.c_int64(0) for _ in range(4)]
        _capi.call("cl_tree_columns_layout", geo, 1, *[ctypes.byref(i) for i in v])
        assert v[0].value == 1 and v[1].value == xw.shape[0] and v[2].value == ref.shape[0]
        cols = 2 * words
        x32 = xw.view(torch.int32)
        colmaj = torch.empty((cols, xw.shape[0]), dtype=torch.int32, device=device)
        s = torch.cuda.current_stream().cuda_stream
        _capi.call("cl_packed_rows_to_columns", x32.data_ptr(), colmaj.data_ptr(), xw.shape[0],
                   cols * 4, xw.shape[0], s)
        assert torch.equal(colmaj, x32.t())
        tables = torch.empty(v[3].value, dtype=torch.int32, device=device)
        out = torch.empty((cols, ref.shape[0]), dtype=torch.int32, device=device)
        one = lambda t: (ctypes.c_void_p * 1)(t.data_ptr())
        _capi.call("cl_tree_columns", colmaj.data_ptr(), cols, xw.shape[0], geo, 1, one(gates),
                   one(sel), tables.data_ptr(), out.data_ptr(), ref.shape[0], s)
        assert torch.equal(out.t(), ref.view(torch.int32))
        assert bool((out.t().reshape(cout, -1)[::97] == -1).all())


def test_tree_front_steps_aside(device):
    """Taps outside the kernel window take the layer-by-layer kernels."""
    model = tree_net([(2, 8, 2, 1, 3)], [(32, 100)], 10, 3, device)
    x = cl.PackBitsTensor(torch.rand((100, 2 * 64), device=device) < 0.5, 64)
    net = cl.PackedNetwork(model)
    assert net._call_front(x) is not None
    with torch.no_grad():
        model[0].selection[0, 0] = 7 << 8            # row 7 of a 3 x 3 window
    assert net._call_front(x) is None
    assert torch.equal(net(x), model(cl.PackBitsTensor.from_packed(x.t.clone(), x.pad_len)))


def test_circuit_follows_the_producer(device):
    """A circuit of convolutions and tail stands for the tables it was built from: after a change
    of a convolution's winners the call evaluates the layers as they are."""
    torch.manual_seed(3)
    conv = cl.ConvLayer((3, 40, 40), padding=1, c_out=16, ks=3, stride=2)
    model = torch.nn.Sequential(conv, torch.nn.Flatten(), cl.LogicLayer(conv.out_dim, 3500),
                                cl.GroupSum(10, 1.0)).to(device)
    for m in model:
        if hasattr(m, "freeze"):
            m.freeze()
    model.eval()
    net = cl.PackedNetwork(model)
    assert net.producer is not None and net.circuit is not None
    bits = np.random.default_rng(0).integers(0, 2, (200, 4800)).astype(bool)
    x = cl.PackBitsTensor(torch.as_tensor(bits, device=device), 64)

    def layers():
        return model(cl.PackBitsTensor.from_packed(x.t.clone(), x.pad_len))

    before = net(x)
    assert torch.equal(before, layers())
    conv.w.copy_((conv.w + 1) % conv.num_gates)
    after = net(x)
    assert torch.equal(after, layers()) and not torch.equal(before, after)


@pytest.mark.parametrize("out_dim,k", [(8500, 50), (17000, 200)])
def test_counts_of_more_than_32_classes_past_the_register_tables(device, out_dim, k):
    """A network wider than the register-table kernel takes (a column per workgroup): more
    (sample, class) pairs than threads."""
    model = frozen_net([(64, 17000), (17000, out_dim)], k, 4, k, device)
    rng = np.random.default_rng(k)
    x = cl.PackBitsTensor(torch.as_tensor(rng.integers(0, 2, (130, 64)).astype(bool),
                                          device=device), 64)
    counts = cl.PackedNetwork(model, bank_aware=False)(x)
    assert np.array_equal(np_(counts), oracle_counts(model, np_(x.t).view(np.uint64), 130))


def ran(net, x):
    """(counts, entry points that ran) of a call."""
    from compactlogic_amd import timing
    with timing.record() as rec:
        counts = net(x)
    return counts, {name.split("[")[0] for name in rec.summary()}


def packed_bits(device, n, feats, seed, bits=64):
    rng = np.random.default_rng(seed)
    return cl.PackBitsTensor(torch.as_tensor(rng.integers(0, 2, (n, feats)).astype(bool),
                                             device=device), bits)


@pytest.mark.parametrize("dims,k,g_n,n", [
    ([(40, 64), (64, 60)], 6, 4, 64),                        # a slot per layer
    ([(100, 300), (300, 300), (300, 200)], 10, 16, 1000),
    ([(12, 20)] + [(20, 20)] * 14 + [(20, 30)], 3, 8, 130),  # sixteen layers
    ([(64, 2000), (2000, 1000)], 8, 16, 4096),               # two slots
    ([(100, 4000), (4000, 3000)], 40, 4, 500),               # four; more classes than waves
    ([(3000, 5000), (5000, 2600)], 4, 16, 700),              # eight; 4 inputs per thread
    ([(784, 9000), (9000, 9000)], 3, 4, 200),                # twelve; 47 rows per lane in a count
    ([(64, 15000), (15000, 16000)], 2, 4, 300),              # sixteen
    ([(64, 17000), (17000, 8500)], 10, 4, 200),              # wider than the register tables
    ([(64, 17000), (17000, 8500)], 50, 4, 130),              # there: more than 32 classes
    ([(64, 13000)] + [(13000, 13000)] * 5, 100, 4, 70),      # more layers than registers
])
@pytest.mark.parametrize("bank_aware", [True, False])
def test_row_tables_match_oracle_and_layerwise(device, dims, k, g_n, n, bank_aware):
    """Every row of every layer, in bank-aware places and in row order: the way of the networks
    that no circuit takes."""
    model = frozen_net(dims, k, g_n, sum(d[1] for d in dims), device)
    x = packed_bits(device, n, dims[0][0], n)
    counts, entries = ran(cl.PackedNetwork(model, bank_aware=bank_aware, prune=False), x)
    assert entries == {"cl_packed_network"}
    assert np.array_equal(np_(counts), oracle_counts(model, np_(x.t).view(np.uint64), n))
    assert torch.equal(counts, model(cl.PackBitsTensor.from_packed(x.t.clone(), x.pad_len)))


def test_circuit_is_the_default_where_it_pays(device):
    """Few classes: the circuit; as many as there are rows: every row."""
    for k, entry in ((10, "cl_packed_circuit"), (1000, "cl_packed_network")):
        model = frozen_net([(100, 2000), (2000, 2000)], k, 16, k, device)
        x = packed_bits(device, 500, 100, k)
        counts, entries = ran(cl.PackedNetwork(model), x)
        assert entries == {entry}
        assert np.array_equal(np_(counts), oracle_counts(model, np_(x.t).view(np.uint64), 500))


@pytest.mark.parametrize("in_shape,c_out,convs,widths,k,n,bits", [
    ((4, 16, 16), 32, 1, [4200, 2100], 10, 1000, 64),    # 8 slots, second layer over the input
    ((2, 12, 12), 40, 1, [12000, 10000], 10, 333, 64),   # 16 slots, nothing held
    ((5, 15, 15), 40, 1, [12000, 10000], 20, 100, 32),   # 9000 rows: held slots; odd words
    ((3, 16, 16), 24, 1, [5000, 4000, 2100], 3, 4096, 64),  # three layers
    ((3, 16, 16), 32, 2, [4200, 2100], 100, 1000, 64),   # two convs composed; many classes
    ((4, 16, 16), 24, 3, [3100, 1550], 5, 333, 64),      # conv layer by layer, then a pair
])
@pytest.mark.parametrize("bank_aware", [True, False])
def test_row_tables_on_columns(device, in_shape, c_out, convs, widths, k, n, bits, bank_aware):
    """The producer written column-major and the tail's rows on those columns."""
    model = small_conv_net(device, in_shape, c_out, widths, k, seed=n, convs=convs)
    x = packed_bits(device, n, int(np.prod(in_shape)), n, bits)
    net = cl.PackedNetwork(model, bank_aware=bank_aware, prune=False)
    counts, entries = ran(net, x)
    pair = "cl_eval_packed_indexed" + ("_pair" if convs > 1 else "") + "_columns"
    assert {pair, "cl_packed_network_columns"} <= entries and "cl_packed_circuit" not in entries
    words = np_(x.t)
    if words.dtype != np.int64:                  # 32-bit words: pad to whole 64-bit words
        words = np.concatenate([words, np.zeros((words.shape[0], words.shape[1] % 2),
                                                words.dtype)], 1)
    ref = conv_oracle_counts(model, np.ascontiguousarray(words).view(np.uint64), n)
    assert np.array_equal(np_(counts), ref)


def test_row_tables_of_cfg5(device):
    cfg = configs.CONV_CONFIGS["cfg5"]
    model = configs.conv_network(cfg, device=device)
    configs.freeze_argmax(model)
    xw = configs.packed_input_words(int(np.prod(cfg.in_shape)), 64, device=device)
    counts, entries = ran(cl.PackedNetwork(model, prune=False), xw)
    assert entries == {"cl_eval_packed_indexed_pair_columns", "cl_packed_network_columns"}
    assert np.array_equal(np_(counts), conv_oracle_counts(model, np_(xw).view(np.uint64), 1 << 12))


@pytest.mark.parametrize("side,blocks,dense,k,n", [
    (32, [(3, 40, 2, 1, 3), (40, 32, 2, 1, 3)], [(128, 300), (300, 200)], 10, 1000),
    (16, [(2, 17, 1, 1, 3)], [(1088, 1000), (1000, 990)], 90, 333),
    (32, [(9, 16, 2, 1, 3)], [(1024, 16000), (16000, 16000)], 10, 200),   # held slots
])
def test_row_tables_after_the_tree_front(device, side, blocks, dense, k, n):
    """The tail's rows in the places of the column-major input that the blocks write."""
    model = tree_net(blocks, dense, k, n, device)
    x = packed_bits(device, n, blocks[0][0] * side * side, n)
    counts, entries = ran(cl.PackedNetwork(model, prune=False), x)
    assert entries == {"cl_packed_rows_to_columns", "cl_tree_columns",
                       "cl_packed_network_columns"}
    assert torch.equal(counts, model(cl.PackBitsTensor.from_packed(x.t.clone(), x.pad_len)))


def test_tree_front_needs_whole_words_and_a_square(device):
    """Rows of an odd number of 32-bit words, and a feature count that is no channels * side^2,
    are left to the layer-by-layer kernels, which refuse them."""
    from compactlogic_amd.packed_net import tree_columns_layout
    model = tree_net([(2, 8, 2, 1, 3)], [(32, 100)], 10, 3, device)
    net = cl.PackedNetwork(model)
    for n in (96, 65):                           # three words of 32
        x = packed_bits(device, n, 2 * 64, n, 32)
        assert x.t.shape[1] == 3 and net._call_front(x) is None
        with pytest.raises(RuntimeError, match="multiple of 8"):
            net(x)
    assert net._call_front(packed_bits(device, 128, 2 * 64, 1, 32)) is not None
    assert tree_columns_layout(net.front, 2 * 64) is not None
    assert tree_columns_layout(net.front, 2 * 60) is None and \
        tree_columns_layout(net.front, 129) is None
    with pytest.raises(ValueError, match="non-square"):
        net(packed_bits(device, 64, 2 * 60, 1))


def producer_net(device):
    torch.manual_seed(3)
    conv = cl.ConvLayer((3, 40, 40), padding=1, c_out=16, ks=3, stride=2)
    model = torch.nn.Sequential(conv, torch.nn.Flatten(), cl.LogicLayer(conv.out_dim, 3500),
                                cl.GroupSum(10, 1.0)).to(device)
    return model, conv


def test_circuit_of_a_producer_goes_by_its_winners(device, monkeypatch):
    """New table tensors of the same winners (a layer frozen again, winners that change and come
    back) keep the circuit; the row tables are laid out for the first winners that differ."""
    from compactlogic_amd import packed_net
    model, conv = producer_net(device)
    for m in (conv, model[2]):
        m.freeze()
    model.eval()
    net = cl.PackedNetwork(model)
    x = packed_bits(device, 200, 4800, 0)

    def check(entry, calls=1):
        counts, entries = ran(net, x)
        assert entry in entries and len(entries) == calls
        assert torch.equal(counts, model(cl.PackBitsTensor.from_packed(x.t.clone(), x.pad_len)))

    monkeypatch.setattr(packed_net, "_ROWS_IN_CACHE", 0)   # rows turned to columns first
    check("cl_packed_circuit", 2)
    monkeypatch.undo()
    check("cl_packed_circuit")
    conv.freeze()                                # a new winner tensor
    check("cl_packed_circuit")
    assert net.tables is None
    conv.w.copy_((conv.w + 1) % conv.num_gates)
    check("cl_packed_network_columns", 2)
    check("cl_packed_network_columns", 2)
    conv.freeze()
    check("cl_packed_circuit")


@pytest.mark.parametrize("frozen", [True, False])
def test_changed_producer_under_capture(device, frozen):
    """A graph captured right after a convolution's winners changed, with no call before it,
    counts with the new winners; layers that may still train are read at each replay."""
    model, conv = producer_net(device)
    model[2].freeze()
    if frozen:
        conv.freeze()
    model.eval()
    net = cl.PackedNetwork(model)
    assert net.circuit is not None and (net.tables is None) == frozen
    x = packed_bits(device, 200, 4800, 1)
    warm = cl.PackedNetwork(model, prune=False)(x)         # loads the kernels
    with torch.no_grad():
        if frozen:
            conv.w.copy_((conv.w + 1) % conv.num_gates)
        else:
            conv.weights.copy_(conv.weights.roll(1, 1))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        counts = net(x)
    for _ in range(2):
        counts.zero_()
        graph.replay()
        torch.cuda.synchronize()
        ref = model(cl.PackBitsTensor.from_packed(x.t.clone(), x.pad_len))
        assert torch.equal(counts, ref) and not torch.equal(counts, warm)
        if not frozen:
            with torch.no_grad():
                conv.weights.copy_(conv.weights.roll(1, 1))


def test_copied_network_has_tables_of_its_own(device):
    import copy
    model = frozen_net([(64, 400), (400, 300)], 10, 8, 2, device)
    x = packed_bits(device, 300, 64, 2)
    net = cl.PackedNetwork(model)
    ref = net(x)
    other = copy.deepcopy(net)
    net.circuit.tables.zero_()
    assert other.circuit.tables.data_ptr() != net.circuit.tables.data_ptr()
    assert torch.equal(other(x), ref)


def test_tree_blocks_take_columns_where_they_pay(device):
    """The rule of the column pass: from 32 K samples for many channels of 64 positions, never for
    channels that leave waves idle, positions off 64 or an input of far more rows than outputs;
    both ways count alike on either side of it."""
    from compactlogic_amd.packed_net import tree_columns_from
    wide = tree_net([(9, 256, 2, 1, 3), (256, 512, 2, 1, 3)], [(2048, 2000)], 10, 1, device)
    blocks = [wide[0], wide[1]]
    assert tree_columns_from(blocks, 9 * 1024) == 1024
    for block, rows in (((2, 17, 1, 1, 3), 512), ((3, 10, 1, 1, 3), 432), ((64, 64, 1, 1, 3), 16384)):
        layer = cl.ConvLogicLayer(block[0], block[1], stride=1, padding=1, kernel=3, complete=True,
                                  num_chn=0)
        assert tree_columns_from([layer], rows) == float("inf")
    net = cl.PackedNetwork(wide)
    for n, columns in ((32768 - 64, False), (32768, True)):
        gen = torch.Generator(device=device).manual_seed(n)
        words = torch.randint(-2**62, 2**62, (9 * 1024, n // 64), generator=gen, device=device)
        counts, entries = ran(net, words)
        assert ("cl_tree_columns" in entries) == columns
        assert torch.equal(counts, wide(cl.PackBitsTensor.from_packed(words)))


@pytest.mark.parametrize("prune", [True, False])
def test_rows_off_four_bytes_are_refused_alike(device, prune):
    """Rows that are no whole 32-bit words raise the library's error on either way."""
    from compactlogic_amd._capi import CompactLogicError
    net = cl.PackedNetwork(frozen_net([(64, 400), (400, 300)], 10, 8, 4, device), prune=prune)
    for bits in (8, 16):
        with pytest.raises(CompactLogicError, match="multiple of 4 bytes"):
            net(packed_bits(device, 9, 64, bits, bits))
