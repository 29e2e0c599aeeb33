"""Layers of few channels re-packed with several taps per word, from the fp32 input in one launch (k_dense_rows in
fastertnn_amd/csrc/pack_kernels.hip), and their product on packed rows or the vector ALU: every kind of channel count, words that taps
fill and do not, several groups of words, windows, borders and strides, rows that span images, all types, infinite and NaN
inputs, bit for bit against the oracle, with nothing written past the result."""
import numpy as np
import pytest

from fastertnn_amd import BNN, TYPE_NAMES, act_is_ternary, weight_is_ternary
from tests.cases import ALL_TYPES

pytestmark = pytest.mark.gpu

# (batch, C, IH, IW, KN, KH, KW, padding, stride)
LAYERS = [(1, 9, 5, 7, 3, 3, 3, 1, 1), (4, 12, 13, 13, 58, 1, 5, 0, 1), (3, 16, 9, 11, 64, 3, 3, 1, 2), (2, 21, 6, 6, 33, 3, 3, 2, 1), (5, 17, 4, 9, 16, 5, 5, 2, 3),
          (1, 20, 40, 41, 31, 5, 5, 0, 1), (2, 10, 12, 12, 20, 7, 7, 3, 1), (3, 24, 7, 8, 40, 9, 9, 4, 1), (1, 13, 33, 1, 100, 9, 1, 4, 1), (2, 30, 9, 9, 34, 4, 4, 1, 1),
          (1, 32, 9, 10, 70, 4, 4, 0, 2), (1, 16, 300, 230, 5, 5, 5, 2, 1)]
# the explicit vector-ALU engine takes fewer channels too; one channel fills four words with 256 taps
FEW = [(2, 1, 40, 50, 9, 17, 16, 8, 1), (2, 3, 20, 20, 33, 7, 7, 3, 2), (1, 8, 9, 9, 20, 3, 3, 1, 1), (1, 1, 30, 30, 4, 5, 5, 0, 1)]

# from the input's bit planes (dense_rows_from_input says so of each, tests/test_layer_plans.py): pixels by the hundred thousand or windows that share most of their taps
PLANES = [(26, 17, 63, 63, 8, 11, 11, 0, 2), (5, 19, 41, 47, 10, 13, 13, 0, 1), (9, 24, 60, 61, 20, 9, 9, 4, 2), (13, 32, 90, 91, 33, 4, 4, 2, 2), (3, 9, 99, 120, 17, 17, 17, 8, 3)]
FEW_PLANES = [(4, 3, 120, 121, 9, 11, 11, 5, 2), (1, 1, 300, 300, 4, 17, 17, 0, 2)]


def _check(hip, oracle, typ, layer, engines):
    import torch
    n, c, h, w, kn, kh, kw, pad, stride = layer
    print("case", TYPE_NAMES[typ], layer, flush=True)
    rng = np.random.default_rng(7 + typ + c + kn)
    x = rng.standard_normal((n, c, h, w)).astype(np.float32)
    x.reshape(-1)[:5] = [np.inf, -np.inf, np.nan, 0.0, -0.0]
    thr = np.linspace(0.2, 0.8, n) if act_is_ternary(typ) else np.linspace(-0.3, 0.3, n)
    thr = thr.astype(np.float32)
    wt = weight_is_ternary(typ)
    qw = oracle.pack_weights(rng.standard_normal((kn, c, kh, kw)).astype(np.float32), np.full(kn, 0.5 if wt else 0.0, np.float32), wt)
    want = oracle.conv(typ, x, thr, qw, kn, kh, kw, pad, stride, -0.25)
    x_d, thr_d, qw_d = (torch.from_numpy(v).cuda() for v in (x, thr, np.asarray(qw)))
    for engine in engines:
        out = torch.full((want.size + 64,), float("nan"), device="cuda")
        if engine is None:
            hip.conv_prepared(typ, x_d, thr_d, hip.prepare_conv_weights(typ, qw_d, c, kn, kh, kw), kn, kh, kw, pad, stride, -0.25, out=out)
        else:
            hip.conv(typ, x_d, thr_d, qw_d, kn, kh, kw, pad, stride, -0.25, out=out, engine=engine)
        got = out.cpu().numpy()
        assert got[:want.size].tobytes() == want.tobytes(), engine
        assert np.isnan(got[want.size:]).all()


@pytest.mark.parametrize("typ", ALL_TYPES, ids=lambda t: TYPE_NAMES[t])
@pytest.mark.parametrize("layer", LAYERS, ids=lambda v: "x".join(map(str, v)))
def test_layers(hip, oracle, typ, layer):
    _check(hip, oracle, typ, layer, (None, hip.ENGINE_AUTO, hip.ENGINE_VALU))


@pytest.mark.parametrize("typ", ALL_TYPES, ids=lambda t: TYPE_NAMES[t])
@pytest.mark.parametrize("layer", FEW, ids=lambda v: "x".join(map(str, v)))
def test_fewer_channels_on_the_vector_alu(hip, oracle, typ, layer):
    _check(hip, oracle, typ, layer, (hip.ENGINE_VALU,))


def test_input_of_more_than_4_gib(hip):
    """elements beyond 32 bits of byte offset: the last images against a batch of their own"""
    import torch
    n, c, h, w, kn = 16400, 16, 64, 64, 2
    print("case", n, c, h, w, flush=True)
    g = torch.Generator(device="cuda").manual_seed(2)
    x = torch.randn((n, c, h, w), generator=g, device="cuda")
    qw = hip.pack_weights(torch.randn((kn, c, 3, 3), generator=g, device="cuda"), torch.zeros(kn, device="cuda"), False)
    thr = torch.full((n,), 0.1, device="cuda")
    got = hip.conv(BNN, x, thr, qw, kn, 3, 3, 1, 1, 0.5).reshape(n, -1)
    want = hip.conv(BNN, x[-3:].contiguous(), thr[-3:].contiguous(), qw, kn, 3, 3, 1, 1, 0.5).reshape(3, -1)
    assert torch.equal(got[-3:], want)


@pytest.mark.parametrize("typ,c,kn", [(0, 9, 2), (2, 1, 2), (3, 3, 2), (1, 9, 16)], ids=("tnn9", "btn1", "bnn3", "tbn9"))
def test_more_than_2_to_29_pixels(hip, typ, c, kn):
    """more row blocks than a grid's x takes, inputs on both sides of 4 GiB: the first and the last images against batches of their own"""
    import torch
    n, h, w = 8193, 256, 256
    print("case", TYPE_NAMES[typ], n, c, h, w, kn, flush=True)
    g = torch.Generator(device="cuda").manual_seed(4)
    x = torch.randn((n, c, h, w), generator=g, device="cuda")
    wt = weight_is_ternary(typ)
    qw = hip.pack_weights(torch.randn((kn, c, 3, 3), generator=g, device="cuda"), torch.full((kn,), 0.5 if wt else 0.0, device="cuda"), wt)
    thr = torch.full((n,), 0.4 if act_is_ternary(typ) else 0.1, device="cuda")
    got = hip.conv(typ, x, thr, qw, kn, 3, 3, 1, 1, 0.5).reshape(n, -1)
    for part in (slice(0, 2), slice(n - 2, n)):
        want = hip.conv(typ, x[part].contiguous(), thr[part].contiguous(), qw, kn, 3, 3, 1, 1, 0.5).reshape(2, -1)
        assert torch.equal(got[part], want), part
    del x, got, want
    torch.cuda.empty_cache()


@pytest.mark.parametrize("typ", ALL_TYPES, ids=lambda t: TYPE_NAMES[t])
@pytest.mark.parametrize("layer", PLANES + FEW_PLANES, ids=lambda v: "x".join(map(str, v)))
def test_from_bit_planes(hip, oracle, typ, layer):
    _check(hip, oracle, typ, layer, (None, hip.ENGINE_AUTO, hip.ENGINE_VALU) if layer in PLANES else (hip.ENGINE_VALU,))


@pytest.mark.parametrize("layer", [LAYERS[2], PLANES[0], FEW[0]], ids=("input", "planes", "one channel"))
def test_under_capture(hip, layer):
    """replays between eager work, each on another input"""
    import torch
    n, c, h, w, kn, kh, kw, pad, stride = layer
    print("case", layer, flush=True)
    g = torch.Generator(device="cuda").manual_seed(6)
    x = torch.randn((n, c, h, w), generator=g, device="cuda")
    thr = torch.full((n,), 0.4, device="cuda")
    qw = hip.pack_weights(torch.randn((kn, c, kh, kw), generator=g, device="cuda"), torch.full((kn,), 0.5, device="cuda"), True)
    oh, ow = hip.out_dim(h, pad, kh, stride), hip.out_dim(w, pad, kw, stride)
    out = torch.empty((n, kn, oh, ow), device="cuda")
    scratch = torch.empty(hip.conv_scratch_bytes(0, n, c, h, w, kn, kh, kw, pad, stride), dtype=torch.uint8, device="cuda")
    once = lambda y: hip.conv(0, x, thr, qw, kn, kh, kw, pad, stride, 0.5, scratch=scratch, out=y, engine=hip.ENGINE_VALU)
    once(out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        once(out)
    for rep in range(4):
        x.normal_()
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        want = once(torch.empty_like(out))
        assert torch.equal(out, want), rep
