"""Thresholds of a quantised hand-over as cuts on the integer sum: slopes and thresholds at which the staircase degenerates or
the kernels must compare after PReLU instead (negative slopes and ternary thresholds, infinities), thresholds that sums meet
exactly, for the layer kernel on both tiles and every K split and for the first-layer kernel, bit for bit against the oracle."""
import numpy as np
import pytest

from fastertnn_amd import BNN, BTN, TBN, TNN, TYPE_NAMES, act_is_ternary, synth, weight_is_ternary

pytestmark = pytest.mark.gpu

INF = float("inf")
# (slope of the handing layer, threshold of the taking one)
POINTS = [(0.5, 0.0), (0.5, 3.0), (0.0, 0.0), (0.0, -1.0), (1.0, 2.0), (1.0, -2.5), (-0.5, 1.0), (2.0, 4.0), (1 / 3, 1.0),
          (0.5, -0.5), (1e-30, 1e-30), (0.5, 5000.0), (0.5, INF), (0.5, -INF), (3e38, 1.0)]


def _layer(oracle, typ, row, seed):
    import torch
    wt = weight_is_ternary(typ)
    w = (synth.ternary if wt else synth.binary)(seed, (row[3], row[0], row[5], row[4]))
    qw = oracle.pack_weights(w, np.full(row[3], 0.5 if wt else 0.0, np.float32), wt)
    return qw, torch.from_numpy(qw).cuda()


@pytest.mark.parametrize("typ", (TNN, TBN, BTN, BNN), ids=lambda t: TYPE_NAMES[t])
# tiles of 64 x 64: 6 (the layer runs on 32 x 32), 288 (K split over four wavefronts), 512 (two), 632 (not split)
@pytest.mark.parametrize("first,hw", [(3, 12), (64, 12), (70, 96), (64, 128), (64, 142)],
                         ids=["first-layer", "32x32", "64x64", "64x64-two", "64x64-whole"])
def test_hand_over_thresholds(hip, oracle, typ, first, hw):
    import torch
    for other in (TNN, BNN):
        rows = [(first, hw, hw, 65, 3, 3, 1, 1), (65, hw, hw, 33, 1, 1, 0, 1)]
        types = (typ, other)
        weights = [_layer(oracle, t, r, 40 + i) for i, (t, r) in enumerate(zip(types, rows))]
        x = synth.normal(77, (1, first, hw, hw))
        thr0 = 0.5 if act_is_ternary(typ) else 0.0
        for alpha, thr in POINTS:   # (no infinite slope: 0 * inf is NaN, whose quantisation the reference's own paths disagree on)
            print("case", TYPE_NAMES[typ], TYPE_NAMES[other], first, hw, alpha, thr, flush=True)
            layers = [dict(type=t, shape=r, threshold=th, alpha=a, qw=w[1])
                      for t, r, w, th, a in zip(types, rows, weights, (thr0, thr), (alpha, 0.5))]
            net = hip.Net(1, layers)
            got = net.run(torch.from_numpy(x).cuda()).cpu().numpy()
            net.close()
            want = x
            for l, (qw, _), r in zip(layers, weights, rows):
                want = oracle.conv(l["type"], want, np.full(1, l["threshold"], np.float32), qw, r[3], r[5], r[4], r[6], r[7], l["alpha"])
            assert got.tobytes() == want.tobytes(), (alpha, thr)
