"""Small layers in one launch (fastertnn_amd/csrc/direct_kernels.hip): windows, strides, padding, images smaller than a tile and of
ragged sizes, channel counts around the words of a record, rows of a single word and of many, every split of K, and fully connected
layers of one image to several tiles of them, all types, bit for bit against the vector-ALU engine; then the lines beyond which such
a layer takes two launches, thresholds of every sign and infinite inputs."""
import pytest
import torch

from fastertnn_amd import TYPE_NAMES, act_is_ternary, weight_is_ternary

pytestmark = pytest.mark.gpu

# (batch, C, IH, IW, KN, KH, KW, padding, stride)
LAYERS = [(1, 33, 5, 7, 1, 1, 1, 0, 1), (2, 63, 4, 4, 33, 3, 3, 1, 1), (3, 64, 9, 9, 32, 3, 3, 1, 2), (5, 65, 2, 2, 1000, 1, 1, 0, 2),
          (2, 127, 6, 31, 65, 3, 1, 1, 1), (1, 128, 12, 33, 96, 1, 3, 0, 1), (2, 129, 3, 40, 40, 3, 3, 0, 3), (1, 192, 3, 3, 257, 3, 3, 2, 1),
          (7, 256, 8, 8, 64, 1, 1, 0, 1), (4, 512, 5, 13, 128, 1, 1, 0, 1), (2, 300, 1, 9, 64, 1, 1, 1, 2), (1, 64, 17, 17, 31, 7, 7, 3, 1),
          (60, 40, 8, 8, 256, 3, 3, 0, 1), (24, 64, 14, 14, 256, 3, 3, 1, 1), (1, 64, 2, 200, 64, 5, 3, 2, 1), (16, 40, 16, 16, 64, 3, 5, 1, 1),
          (1, 100, 64, 64, 32, 3, 3, 1, 1), (2, 1024, 1, 3, 90, 1, 1, 0, 1)]
# fully connected: (images, C, KN); rows of C floats that 16-byte loads can and cannot take
FC = [(1, 40, 3), (1, 64, 33), (2, 65, 300), (5, 130, 1000), (8, 512, 1000), (32, 100, 64), (33, 96, 70), (70, 66, 31), (1, 4097, 129), (3, 2052, 2000)]
# on both sides of the lines: workgroups, pieces of input with and without a window, fully connected ones
LINES = [(b, 64, 16, 16, 64, 3, 3, 1, 1) for b in (16, 17, 31, 32, 33, 65)] + [(2, c, 10, 10, 128, 3, 3, 1, 1) for c in (128, 129, 192, 193)] + \
        [(4, c, 8, 8, 64, 1, 1, 0, 1) for c in (512, 513)] + [(1, 128, 53, 53, k, 3, 3, 1, 1) for k in (64, 256)]
FC_LINES = [(3, c, 77) for c in (4096, 4097, 4160)] + [(17, 700, 12800), (17, 700, 12801), (1, 2752, 12190), (1, 2752, 12194)]

# every split of K (2^lgS wavefronts on one) with one workgroup per tile and several, windows and none; tests/test_layer_plans.py holds each to its split
SPLITS = {(2, 200, 4, 7, 31, 3, 3, 0, 1): (3, 1), (2, 200, 4, 7, 70, 3, 3, 0, 1): (3, 3), (2, 130, 6, 31, 20, 3, 1, 1, 1): (2, 1), (3, 100, 12, 13, 100, 3, 3, 1, 1): (2, 2),
          (8, 128, 28, 28, 100, 3, 3, 1, 1): (1, 1), (60, 40, 8, 8, 250, 3, 3, 0, 1): (1, 2), (24, 64, 14, 13, 250, 3, 3, 1, 1): (0, 1), (20, 60, 12, 12, 500, 1, 1, 0, 1): (0, 2),
          (20, 130, 9, 9, 270, 1, 1, 0, 1): (1, 3)}
# left to two launches: a single pixel per tile, runs of 10 pairs of K words and more, or of five where a tile has several workgroups
BEYOND = [(26, 40, 3, 3, 1810, 3, 3, 0, 1), (26, 224, 3, 6, 1429, 3, 5, 0, 2), (17, 95, 5, 5, 1045, 3, 3, 1, 1), (4, 79, 12, 12, 864, 3, 3, 1, 1), (24, 47, 6, 6, 600, 5, 5, 2, 1)]


def _run(hip, typ, layer, alpha, thr=None, x=None, aligned=True):
    n, c, h, w, kn, kh, kw, pad, stride = layer
    g = torch.Generator(device="cuda").manual_seed(3 + typ + n + c + h * w + kn)
    wt = weight_is_ternary(typ)
    if x is None:
        x = torch.randn((n, c, h, w), generator=g, device="cuda")
    if not aligned:   # an input that no 16-byte load may take
        x = torch.cat([x.new_zeros(1), x.reshape(-1)])[1:].view(x.shape)
        assert x.data_ptr() % 16 == 4
    if thr is None:
        thr = torch.linspace(0.2, 0.8, n, device="cuda") if act_is_ternary(typ) else torch.linspace(-0.3, 0.3, n, device="cuda")
    qw = hip.pack_weights(torch.randn((kn, c, kh, kw), generator=g, device="cuda"), torch.full((kn,), 0.5 if wt else 0.0, device="cuda"), wt)
    oh, ow = hip.out_dim(h, pad, kh, stride), hip.out_dim(w, pad, kw, stride)
    prepared = hip.prepare_conv_weights(typ, qw, c, kn, kh, kw)
    size = n * kn * oh * ow
    want = hip.conv(typ, x, thr, qw, kn, kh, kw, pad, stride, alpha, engine=hip.ENGINE_VALU).reshape(-1)
    for how in ("prepared", "packed"):
        out = torch.full((size + 64,), float("nan"), device="cuda")
        if how == "prepared":
            hip.conv_prepared(typ, x, thr, prepared, kn, kh, kw, pad, stride, alpha, out=out)
        else:
            hip.conv(typ, x, thr, qw, kn, kh, kw, pad, stride, alpha, out=out, engine=hip.ENGINE_MFMA_F4)
        assert torch.equal(out[:size].view(torch.int32), want.view(torch.int32)), how
        assert bool(torch.isnan(out[size:]).all()), how


@pytest.mark.parametrize("typ", range(4), ids=[TYPE_NAMES[t] for t in range(4)])
@pytest.mark.parametrize("layer", LAYERS + LINES + list(SPLITS) + BEYOND, ids=lambda v: "x".join(map(str, v)))
def test_layers(hip, typ, layer):
    print("case", TYPE_NAMES[typ], layer, flush=True)
    _run(hip, typ, layer, -0.25)


@pytest.mark.parametrize("typ", range(4), ids=[TYPE_NAMES[t] for t in range(4)])
@pytest.mark.parametrize("layer", FC + FC_LINES, ids=lambda v: "x".join(map(str, v)))
def test_fully_connected(hip, typ, layer):
    print("case", TYPE_NAMES[typ], layer, flush=True)
    n, c, kn = layer
    for aligned in (True, False):
        _run(hip, typ, (n, c, 1, 1, kn, 1, 1, 0, 1), 0.5, aligned=aligned)


@pytest.mark.parametrize("typ", range(4), ids=[TYPE_NAMES[t] for t in range(4)])
@pytest.mark.parametrize("layer", [(4, 70, 6, 5, 40, 3, 3, 1, 1), (4, 70, 1, 1, 40, 1, 1, 0, 1)], ids=("window", "fc"))
def test_thresholds_and_infinities(hip, typ, layer):
    """thresholds that are negative (below -t comes first), zero of either sign and infinite; inputs on the threshold, infinite, -0"""
    n, c, h, w = layer[:4]
    thr = torch.tensor([-0.5, 0.0, -0.0, float("inf")], device="cuda")
    x = torch.randint(-2, 3, (n, c, h, w), device="cuda").float() * 0.25
    x[:, 0], x[:, 1], x[:, 2, 0] = float("inf"), float("-inf"), -0.0
    _run(hip, typ, layer, -0.0, thr=thr, x=x)
    _run(hip, typ, layer, 3.0, thr=-thr, x=x)


def test_under_capture(hip, oracle):
    """replays between eager work, each on another input"""
    from fastertnn_amd import TNN
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn((3, 96, 9, 9), generator=g, device="cuda")
    thr = torch.full((3,), 0.5, device="cuda")
    qw = hip.pack_weights(torch.randn((70, 96, 3, 3), generator=g, device="cuda"), torch.full((70,), 0.5, device="cuda"), True)
    prep = hip.prepare_conv_weights(TNN, qw, 96, 70, 3, 3)
    out = torch.empty((3, 70, 9, 9), device="cuda")
    scratch = torch.empty(hip.conv_scratch_bytes(TNN, 3, 96, 9, 9, 70, 3, 3, 1, 1), dtype=torch.uint8, device="cuda")
    once = lambda: hip.conv_prepared(TNN, x, thr, prep, 70, 3, 3, 1, 1, 0.5, scratch=scratch, out=out)
    once()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        once()
    for rep in range(4):
        x.normal_()
        out.zero_()
        graph.replay()
        want = hip.conv(TNN, x, thr, qw, 70, 3, 3, 1, 1, 0.5, engine=hip.ENGINE_VALU)
        torch.cuda.synchronize()
        assert torch.equal(out, want), rep


@pytest.mark.parametrize("typ", range(4), ids=[TYPE_NAMES[t] for t in range(4)])
@pytest.mark.parametrize("layer", [(8, 128, 28, 28, 128, 3, 3, 1, 1), (4, 64, 16, 16, 64, 1, 1, 0, 1), (8, 512, 1, 1, 512, 1, 1, 0, 1), (8, 40, 1, 1, 300, 1, 1, 0, 1)],
                         ids=lambda v: "x".join(map(str, v)))
def test_result_over_its_input(hip, typ, layer):
    """the result in the place of the input, over a part of it at either end, and over the thresholds: as in a place of its own"""
    n, c, h, w, kn, kh, kw, pad, stride = layer
    print("case", TYPE_NAMES[typ], layer, flush=True)
    g = torch.Generator(device="cuda").manual_seed(9 + typ)
    wt = weight_is_ternary(typ)
    values = torch.randn((n, c, h, w), generator=g, device="cuda")
    thr0 = torch.linspace(0.2, 0.8, n, device="cuda") if act_is_ternary(typ) else torch.linspace(-0.3, 0.3, n, device="cuda")
    qw = hip.pack_weights(torch.randn((kn, c, kh, kw), generator=g, device="cuda"), torch.full((kn,), 0.5 if wt else 0.0, device="cuda"), wt)
    prep = hip.prepare_conv_weights(typ, qw, c, kn, kh, kw)
    want = hip.conv_prepared(typ, values, thr0, prep, kn, kh, kw, pad, stride, 0.5)
    nx, ny = values.numel(), want.numel()
    lead = max(nx, ny)
    for at in (0, nx // 2, -(ny // 2), nx - 1, 1 - ny, None):   # the result's place, from the input's; None: over the thresholds
        buf = torch.zeros(nx + 2 * lead + n, device="cuda")
        x, thr = buf[lead:lead + nx].view(values.shape), buf[-n:]
        x.copy_(values), thr.copy_(thr0)
        y0 = lead + at if at is not None else buf.numel() - ny
        out = buf[y0:y0 + ny].view(want.shape)
        hip.conv_prepared(typ, x, thr, prep, kn, kh, kw, pad, stride, 0.5, out=out)
        assert torch.equal(out, want), at
