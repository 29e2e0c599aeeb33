"""Fully connected layers (1 x 1 kernels on one pixel per image), which run as a product of packed rows from 65 channels on:
every type at ragged sizes, weights packed or prepared, explicit engine and AUTO, with nothing written past the scratch, the
prepared weights or the result, bit for bit against the oracle.  One-pixel layers with padding keep the layer kernels."""
import numpy as np
import pytest

from fastertnn_amd import BNN, TNN, TYPE_NAMES, weight_is_ternary
from tests.cases import ALL_TYPES, make_layer

pytestmark = pytest.mark.gpu

# (images, channels, kernels, padding, stride): one word and two, K tails of 1 to 4 words, tiles of every size, padding
# that leaves one output pixel (which reads the fill)
SHAPES = [(3, 64, 5, 0, 1), (1, 65, 1, 0, 1), (5, 128, 33, 0, 2), (8, 200, 1000, 0, 1), (33, 257, 31, 0, 3),
          (129, 1000, 65, 0, 1), (700, 256, 300, 0, 1), (65, 16384, 100, 0, 1), (2, 200, 40, 1, 3)]


def _guarded(elems, dtype, guard):
    import torch
    return torch.full((elems + 256,), guard, dtype=dtype, device="cuda")


@pytest.mark.parametrize("typ", ALL_TYPES, ids=lambda t: TYPE_NAMES[t])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_fully_connected_layers(hip, oracle, typ, shape):
    import torch
    n, c, kn, pad, stride = shape
    print("case", TYPE_NAMES[typ], shape, flush=True)
    L = make_layer(typ, (c, 1, 1, kn, 1, 1, pad, stride), n, seed=7000 + 31 * n + c + typ)
    L["x"][0, 0], L["x"][-1, -1] = np.inf, -np.inf
    qw = oracle.pack_weights(L["w"], L["wthr"], weight_is_ternary(typ))
    x, thr, qw_d = (torch.from_numpy(np.ascontiguousarray(v)).cuda() for v in (L["x"], L["thr"], qw))
    scratch_bytes = hip.conv_scratch_bytes(typ, n, c, 1, 1, kn, 1, 1, pad, stride)
    weight_bytes = hip._L.ftnn_conv_weights_bytes(typ, c, kn, 1, 1)
    prepared = _guarded(weight_bytes, torch.uint8, 0x5A)
    assert hip._L.ftnn_conv_prepare_weights(typ, qw_d.data_ptr(), c, kn, 1, 1, prepared.data_ptr(), hip._stream()) == 0
    for alpha in (0.5, -0.25):
        want = oracle.conv(typ, L["x"], L["thr"], qw, kn, 1, 1, pad, stride, alpha)
        for how in ("packed", "engine", "prepared"):
            scratch, y = _guarded(scratch_bytes, torch.uint8, 0x5A), _guarded(n * kn, torch.float32, float("nan"))
            if how == "prepared":
                hip.conv_prepared(typ, x, thr, prepared, kn, 1, 1, pad, stride, alpha, scratch=scratch, out=y)
            else:
                hip.conv(typ, x, thr, qw_d, kn, 1, 1, pad, stride, alpha, scratch=scratch, out=y,
                         engine=hip.ENGINE_AUTO if how == "packed" else hip.ENGINE_MFMA_F4)
            got = y.cpu().numpy()
            assert got[:n * kn].tobytes() == want.tobytes(), (how, alpha)
            assert np.isnan(got[n * kn:]).all(), how
            assert bool((scratch[scratch_bytes:] == 0x5A).all()), how
    assert bool((prepared[weight_bytes:] == 0x5A).all())


@pytest.mark.parametrize("typ", (TNN, BNN), ids=lambda t: TYPE_NAMES[t])
def test_prepare_and_layer_under_capture(hip, oracle, typ):
    """weights prepared and the layer run inside one captured graph, replayed on new inputs between eager work"""
    import torch
    n, c, kn = 9, 300, 77
    L = make_layer(typ, (c, 1, 1, kn, 1, 1, 0, 1), n, seed=8100 + typ)
    qw = oracle.pack_weights(L["w"], L["wthr"], weight_is_ternary(typ))
    x, thr, qw_d = (torch.from_numpy(np.ascontiguousarray(v)).cuda() for v in (L["x"], L["thr"], qw))
    y = torch.empty(n * kn, device="cuda")
    scratch = torch.empty(hip.conv_scratch_bytes(typ, n, c, 1, 1, kn, 1, 1, 0, 1), dtype=torch.uint8, device="cuda")

    def once():
        w = hip.prepare_conv_weights(typ, qw_d, c, kn, 1, 1)
        hip.conv_prepared(typ, x, thr, w, kn, 1, 1, 0, 1, 0.5, scratch=scratch, out=y)
    once()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        once()
    for rep in range(4):
        inp = np.roll(L["x"], rep, axis=1)
        x.copy_(torch.from_numpy(np.ascontiguousarray(inp)))
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        want = oracle.conv(typ, inp, L["thr"], qw, kn, 1, 1, 0, 1, 0.5)
        assert y.cpu().numpy().tobytes() == want.tobytes(), rep
