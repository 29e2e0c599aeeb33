"""Layers of few tiles and long rows, whose K is split over eight wavefronts (k_conv_f4 with S = 8 in fastertnn_amd/csrc/mfma_kernels.hip):
either side of the lines (75 words, 256 tiles of 32 x 32), shares of K of every remainder, ragged pixels and kernels, borders and
strides, all types, bit for bit against the vector-ALU engine, with nothing written past the result."""
import pytest

from fastertnn_amd import TYPE_NAMES
from tests.test_gpu_direct import _run

pytestmark = pytest.mark.gpu

# (batch, C, IH, IW, KN, KH, KW, padding, stride)
LAYERS = [(1, 512, 7, 7, 33, 3, 3, 1, 1), (1, 520, 7, 7, 33, 3, 3, 1, 1), (3, 200, 5, 9, 95, 5, 5, 2, 1), (2, 250, 6, 6, 70, 7, 7, 3, 2), (1, 256, 13, 13, 40, 9, 9, 4, 1),
          (5, 4800, 2, 2, 31, 1, 1, 0, 1), (5, 4737, 2, 2, 31, 1, 1, 0, 1), (5, 4736, 2, 2, 31, 1, 1, 0, 1), (17, 330, 6, 6, 65, 5, 5, 0, 1), (1, 700, 1, 8, 1, 1, 7, 3, 1),
          # 239, 256 and 258 tiles
          (1, 257, 85, 96, 32, 4, 4, 0, 1), (1, 257, 128, 64, 32, 5, 5, 2, 1), (1, 257, 131, 63, 20, 5, 5, 2, 1)]


@pytest.mark.parametrize("typ", range(4), ids=[TYPE_NAMES[t] for t in range(4)])
@pytest.mark.parametrize("layer", LAYERS, ids=lambda v: "x".join(map(str, v)))
def test_deep_layers(hip, typ, layer):
    print("case", TYPE_NAMES[typ], layer, flush=True)
    _run(hip, typ, layer, -0.25)
