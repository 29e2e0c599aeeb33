"""Conv layers on the tile kernel with implicit im2row (workgroup tiles whose activation records are gathered from the
quantised input, for strided layers with many tiles, long rows and an fp32 result): forced onto small and ragged layers of
every type with both tile sizes (child processes: the switches are read once per process), and at sizes that take the
route by themselves, as single calls and as chains.  Every result bit for bit against the oracle, where that would take long on
some of the images, and on all of them against the vector-ALU engine."""
import os
import subprocess
import sys

import numpy as np
import pytest

from fastertnn_amd import TNN, TYPE_NAMES, weight_is_ternary
from tests.cases import ALL_TYPES, make_layer

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

_CHILD = r"""
import sys
import numpy as np, torch
sys.path.insert(0, sys.argv[1])
import fastertnn_amd.lib as hip
from fastertnn_amd import TYPE_NAMES, weight_is_ternary
from oracle.ftnn_oracle import Oracle
from tests.cases import make_layer
oracle = Oracle()
# (C, IH, IW, KN, KW, KH, pad, stride), batch: tiles that straddle images, ragged pixel and kernel counts, channel
# tails, strides, windows that are not square, 1 x 1, padding wider than one pixel, rows of 1 .. 50 words (padding words)
SHAPES = [((64, 12, 12, 64, 3, 3, 1, 1), 3), ((130, 17, 17, 70, 3, 3, 1, 2), 5), ((200, 6, 7, 33, 1, 1, 0, 1), 9),
          ((96, 9, 11, 257, 5, 3, 2, 1), 2), ((320, 15, 23, 320, 3, 3, 1, 2), 2), ((64, 30, 30, 300, 3, 3, 1, 1), 1),
          ((128, 8, 8, 130, 2, 2, 0, 2), 7), ((640, 5, 5, 40, 3, 3, 2, 1), 4)]
for typ in range(4):
    for shape, batch in SHAPES:
        L = make_layer(typ, shape, batch, seed=9100 + typ)
        print("case", TYPE_NAMES[typ], shape, batch, flush=True)
        wt = weight_is_ternary(typ)
        qw = oracle.pack_weights(L["w"], L["wthr"], wt)
        for alpha in (0.5, -0.25):
            want = oracle.conv(typ, L["x"], L["thr"], qw, L["kn"], L["kh"], L["kw"], L["pad"], L["stride"], alpha)
            y = torch.full(want.shape, float("nan"), device="cuda")
            hip.conv(typ, torch.from_numpy(L["x"]).cuda(), torch.from_numpy(L["thr"]).cuda(), torch.from_numpy(qw).cuda(),
                     L["kn"], L["kh"], L["kw"], L["pad"], L["stride"], alpha, engine=hip.ENGINE_MFMA_F4, out=y)
            assert y.cpu().numpy().tobytes() == want.tobytes(), (typ, shape, alpha)
print("child ok")
"""


@pytest.mark.parametrize("tile", ["22", "42"])
def test_tile_route_forced_on_small_and_ragged_layers(tile):
    """tiles of 128 kernels x 128 pixels and 256 x 128"""
    env = dict(os.environ, FTNN_CONV_TILES_FROM="1", FTNN_CONV_TILE_SHAPE=tile)
    print("case conv tile route forced, tile shape", tile, flush=True)
    r = subprocess.run([sys.executable, "-c", _CHILD, ROOT], env=env, capture_output=True, text=True, timeout=280)
    assert r.returncode == 0 and "child ok" in r.stdout, r.stdout[-2000:] + r.stderr[-2000:]


@pytest.mark.parametrize("typ", ALL_TYPES, ids=lambda t: TYPE_NAMES[t])
@pytest.mark.parametrize("batch", [13, 8], ids=["batch_13", "batch_8"])
def test_large_layer_without_a_stride(hip, oracle, typ, batch):
    """128 channels, 28 x 28, 256 kernels, rows of 18 words: large, but at stride 1 (the layer kernel), whole call and host call"""
    import torch
    shape = (128, 28, 28, 256, 3, 3, 1, 1)
    assert hip.conv_scratch_bytes(typ, batch, 128, 28, 28, 256, 3, 3, 1, 1) > 0
    L = make_layer(typ, shape, batch, seed=9300 + typ)
    print("case", TYPE_NAMES[typ], shape, batch, flush=True)
    qw = oracle.pack_weights(L["w"], L["wthr"], weight_is_ternary(typ))
    want = oracle.conv(typ, L["x"], L["thr"], qw, L["kn"], 3, 3, 1, 1, 0.5)
    got = hip.conv(typ, torch.from_numpy(L["x"]).cuda(), torch.from_numpy(L["thr"]).cuda(), torch.from_numpy(qw).cuda(),
                   L["kn"], 3, 3, 1, 1, 0.5)
    assert got.cpu().numpy().tobytes() == want.tobytes()
    got = hip.host_conv(typ, L["x"], L["thr"], qw, L["kn"], 3, 3, 1, 1, 0.5)
    assert got.tobytes() == want.tobytes()


def tile_shape(shape, batch):
    """(kernels, pixels) of the workgroup tile that a layer with prepared thresholds and fp32 result runs on, None: the layer kernel"""
    c, ih, iw, kn, kw, kh, pad, stride = shape
    m = batch * ((ih + 2 * pad - kh) // stride + 1) * ((iw + 2 * pad - kw) // stride + 1)
    if stride < 2 or (c + 63) // 64 * kw * kh < 100 or m < 512 or (m + 63) // 64 * ((kn + 63) // 64) < 1500:
        return None
    return (256, 128) if 180 <= (m + 127) // 128 * ((kn + 255) // 256) <= 256 else (128, 128)


@pytest.mark.parametrize("typ", ALL_TYPES, ids=lambda t: TYPE_NAMES[t])
@pytest.mark.parametrize("kn,batch,tile", [(1000, 16, (256, 128)), (300, 48, (128, 128))], ids=["256x128", "128x128"])
def test_layer_that_takes_the_tile_route_by_itself(hip, oracle, typ, kn, batch, tile):
    """256 channels, 40 x 40, 5 x 5 stride 2 (rows of 100 words), 1600 and 1500 tiles of 64 x 64: unprepared and prepared weights, and
    the host call"""
    import torch
    shape = (256, 40, 40, kn, 5, 5, 2, 2)
    assert tile_shape(shape, batch) == tile
    L = make_layer(typ, shape, batch, seed=9400 + typ)
    print("case", TYPE_NAMES[typ], shape, batch, flush=True)
    qw = oracle.pack_weights(L["w"], L["wthr"], weight_is_ternary(typ))
    x, thr, qw_d = torch.from_numpy(L["x"]).cuda(), torch.from_numpy(L["thr"]).cuda(), torch.from_numpy(qw).cuda()
    want = hip.conv(typ, x, thr, qw_d, kn, 5, 5, 2, 2, 0.5, engine=hip.ENGINE_VALU).cpu().numpy()
    for i in (0, batch // 2, batch - 1):
        one = oracle.conv(typ, L["x"][i:i + 1], L["thr"][i:i + 1], qw, kn, 5, 5, 2, 2, 0.5)
        assert want[i:i + 1].tobytes() == one.tobytes(), i
    got = hip.conv(typ, x, thr, qw_d, kn, 5, 5, 2, 2, 0.5)
    assert got.cpu().numpy().tobytes() == want.tobytes()
    got = hip.conv_prepared(typ, x, thr, hip.prepare_conv_weights(typ, qw_d, 256, kn, 5, 5), kn, 5, 5, 2, 2, 0.5)
    assert got.cpu().numpy().tobytes() == want.tobytes()
    assert hip.host_conv(typ, L["x"], L["thr"], qw, kn, 5, 5, 2, 2, 0.5).tobytes() == want.tobytes()


@pytest.mark.parametrize("typ", ALL_TYPES, ids=lambda t: TYPE_NAMES[t])
def test_single_layer_chain(hip, oracle, typ):
    """a chain of one large layer (fp32 in, fp32 out) goes through the same routes from ftnn_net_run: the layer kernel at stride 1 and
    with rows of 36 words, at batch 50 in the net's two half-batch chains; workgroup tiles at stride 2 with rows of 100 words, from
    batch 48 on on both halves"""
    import torch
    for shape, batch, tile in (((128, 28, 28, 256, 3, 3, 1, 1), 13, None), ((256, 30, 30, 300, 3, 3, 1, 2), 50, None),
                               ((256, 40, 40, 1000, 5, 5, 2, 2), 16, (256, 128)), ((256, 40, 40, 640, 5, 5, 2, 2), 48, (256, 128))):
        part = batch if batch < 48 else batch // 2
        assert tile_shape(shape, part) == tile
        L = make_layer(typ, shape, batch, seed=9500 + typ)
        print("case", TYPE_NAMES[typ], shape, batch, flush=True)
        qw = oracle.pack_weights(L["w"], L["wthr"], weight_is_ternary(typ))
        thr = float(L["thr"][0])
        x, qw_d = torch.from_numpy(L["x"]).cuda(), torch.from_numpy(qw).cuda()
        net = hip.Net(batch, [dict(type=typ, shape=shape, threshold=thr, alpha=0.5, qw=qw_d)])
        got = net.run(x)
        net.close()
        tail = (L["kn"], L["kh"], L["kw"], L["pad"], L["stride"], 0.5)
        assert torch.equal(got, hip.conv(typ, x, torch.full((batch,), thr, device="cuda"), qw_d, *tail, engine=hip.ENGINE_VALU))
        some = [0, part - 1, part % batch, batch - 1]
        want = oracle.conv(typ, np.ascontiguousarray(L["x"][some]), np.full(len(some), thr, np.float32), qw, *tail)
        assert got.cpu().numpy()[some].tobytes() == np.ascontiguousarray(want).tobytes()
