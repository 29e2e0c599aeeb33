"""Layer operands at two bits per lane: a pair of K words per load, the two words being planes of one tap (an even number of
64-channel words) or any neighbours (an odd number), the last pair of an odd K half empty; on the layer kernel, split
ways and whole, and behind both quantiser tiles.  Bit for bit against the oracle."""
import numpy as np
import pytest

from fastertnn_amd import TYPE_NAMES, weight_is_ternary
from tests.cases import make_layer

pytestmark = pytest.mark.gpu

# (C, IH, IW, KN, KW, KH, pad, stride), batch: 1, 2, 3 and 5 words of channels, 1 to 9 taps in windows of one column, one row and both,
# every K from one word on, ragged kernel counts; images of small and of ragged sizes; the last three have 290, 522 and
# 2376 tiles of 64 x 64, an odd number of words or of pairs, and the very last is quantised by the larger workgroups
SHAPES = [((64, 9, 7, 40, 1, 1, 0, 1), 2), ((64, 9, 7, 40, 1, 3, 1, 1), 2), ((64, 9, 7, 70, 2, 1, 1, 1), 3), ((64, 11, 11, 64, 3, 3, 1, 2), 3),
          ((128, 9, 9, 33, 3, 3, 1, 1), 2), ((130, 8, 9, 65, 1, 1, 0, 1), 2), ((130, 8, 9, 65, 3, 3, 1, 1), 2), ((190, 5, 5, 96, 2, 2, 0, 1), 4),
          ((300, 6, 6, 100, 1, 1, 0, 1), 3), ((300, 6, 6, 34, 3, 1, 2, 1), 1), ((257, 3, 3, 20, 3, 3, 0, 1), 5),
          ((192, 30, 30, 640, 3, 3, 1, 1), 2), ((320, 44, 44, 1090, 2, 2, 0, 1), 1), ((1030, 17, 16, 1090, 1, 1, 0, 1), 31)]


@pytest.mark.parametrize("typ", range(4), ids=[TYPE_NAMES[t] for t in range(4)])
@pytest.mark.parametrize("shape,batch", SHAPES)
def test_pairs_of_words(hip, oracle, typ, shape, batch):
    import torch
    layer = make_layer(typ, shape, batch, seed=9100 + typ)
    print("case", TYPE_NAMES[typ], shape, batch, flush=True)
    qw = oracle.pack_weights(layer["w"], layer["wthr"], weight_is_ternary(typ))
    want = oracle.conv(typ, layer["x"], layer["thr"], qw, layer["kn"], layer["kh"], layer["kw"], layer["pad"], layer["stride"], 0.5)
    got = hip.conv(typ, torch.from_numpy(layer["x"]).cuda(), torch.from_numpy(np.asarray(layer["thr"])).cuda(), torch.from_numpy(qw).cuda(),
                   layer["kn"], layer["kh"], layer["kw"], layer["pad"], layer["stride"], 0.5, engine=hip.ENGINE_MFMA_F4)
    assert got.cpu().numpy().tobytes() == want.tobytes()
