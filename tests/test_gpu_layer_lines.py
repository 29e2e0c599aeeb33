"""fp32 results of the layer kernel on both sides of every line of its choice (small tiles, K splits, the way a result beyond the
Infinity Cache leaves), bit for bit against the vector-ALU engine."""
import pytest
import torch

from fastertnn_amd import TYPE_NAMES, act_is_ternary, weight_is_ternary

pytestmark = pytest.mark.gpu

# (batch, C, IH, IW, KN, window): tiles of 64 x 64 are IH * IW / 64 here.  9 words per row: lines at 300, 520, 1024; 45: 300, 800, 1500;
# 126: 150; then 264 MiB results of rows that are whole sectors and that are not, the last with one pixel past a tile
LAYERS = [(1, 64, t, 64, 64, 3) for t in (299, 300, 519, 520, 1023, 1024)] + [(1, 320, t, 64, 64, 3) for t in (299, 300, 799, 800, 1499, 1500)] + \
         [(1, 896, t, 64, 64, 3) for t in (149, 150)] + [(2, 64, 256, 256, 530, 1), (2, 64, 255, 255, 535, 1), (2, 64, 1, 65537, 530, 1)]
# 72 words: between 190 and 256 tiles on tiles of 64 x 64, outside and where the last one would be half empty on 32 x 32
LAYERS += [(1, 512, t, 64, 64, 3) for t in (189, 190, 256, 257)] + [(1, 512, 64, 95, 90, 3)]
# few pixels and many kernels, on both sides of the 256 pixels from which they run as im2row + GEMM
LAYERS += [(1, 512, 16, 16, 16384, 3), (1, 512, 1, 257, 11000, 3)]


# stride 2, 108 words: on both sides of the 1500 tiles from which such a layer runs as workgroup tiles, on both of their shapes; then
# results of more than 4 Mi values whose rows are no whole sectors, on both shapes
STRIDED = [(1, 768, 185, 127, 1000, 3), (1, 768, 189, 127, 1000, 3), (1, 768, 299, 255, 300, 3), (5, 768, 75, 71, 1000, 3), (8, 768, 75, 71, 1000, 3)]


@pytest.mark.parametrize("typ", range(4), ids=[TYPE_NAMES[t] for t in range(4)])
@pytest.mark.parametrize("layer", STRIDED, ids=lambda v: "x".join(map(str, v)))
def test_strided_lines(hip, typ, layer):
    n, c, h, w, kn, k = layer
    print("case", TYPE_NAMES[typ], layer, flush=True)
    g = torch.Generator(device="cuda").manual_seed(17 + typ)
    wt = weight_is_ternary(typ)
    x = torch.randn((n, c, h, w), generator=g, device="cuda")
    thr = torch.full((n,), 0.5 if act_is_ternary(typ) else 0.0, device="cuda")
    qw = hip.pack_weights(torch.randn((kn, c, k, k), generator=g, device="cuda"), torch.full((kn,), 0.5 if wt else 0.0, device="cuda"), wt)
    got = hip.conv(typ, x, thr, qw, kn, k, k, 1, 2, -0.25, engine=hip.ENGINE_MFMA_F4)
    want = hip.conv(typ, x, thr, qw, kn, k, k, 1, 2, -0.25, engine=hip.ENGINE_VALU)
    assert torch.equal(got.view(torch.int32), want.view(torch.int32))


@pytest.mark.parametrize("typ", range(4), ids=[TYPE_NAMES[t] for t in range(4)])
@pytest.mark.parametrize("layer", LAYERS, ids=lambda v: "x".join(map(str, v)))
def test_lines(hip, typ, layer):
    n, c, h, w, kn, k = layer
    print("case", TYPE_NAMES[typ], layer, flush=True)
    g = torch.Generator(device="cuda").manual_seed(7 + typ)
    wt = weight_is_ternary(typ)
    x = torch.randn((n, c, h, w), generator=g, device="cuda")
    thr = torch.full((n,), 0.5 if act_is_ternary(typ) else 0.0, device="cuda")
    wf = torch.randn((kn, c, k, k), generator=g, device="cuda")
    qw = hip.pack_weights(wf, torch.full((kn,), 0.5 if wt else 0.0, device="cuda"), wt)
    out = torch.full((n, kn, h, w), float("nan"), device="cuda")
    got = hip.conv(typ, x, thr, qw, kn, k, k, k // 2, 1, -0.25, engine=hip.ENGINE_MFMA_F4, out=out)
    want = hip.conv(typ, x, thr, qw, kn, k, k, k // 2, 1, -0.25, engine=hip.ENGINE_VALU)
    assert torch.equal(got.view(torch.int32), want.view(torch.int32))
