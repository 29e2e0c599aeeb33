"""PReLU slopes at which two ways to write the same function part: a negative zero gives a zero sum the sign the reference's
form for the type gives it (src/tnns/mm_p2_final_tnn_avx2.c:204-208: -0 for TNN; mm_p2_final_tbn_avx2.c:73: +0 for the
others), a positive zero and one leave PReLU at the edges of its maximum form, slopes above one and below zero have none.
Layers with an fp32 result on every tile and K split of the layer kernel, bit for bit against the oracle."""
import numpy as np
import pytest

from fastertnn_amd import TYPE_NAMES, weight_is_ternary
from tests.cases import ALL_TYPES, make_layer

pytestmark = pytest.mark.gpu

# images of 28 x 28, 64 -> 100 channels, 3 x 3: 26 tiles of 64 x 64 (runs on 32 x 32), 196 (K over four wavefronts), 466 (two), 638 (one)
BATCHES = (1, 8, 19, 26)


@pytest.mark.parametrize("typ", ALL_TYPES, ids=lambda t: TYPE_NAMES[t])
@pytest.mark.parametrize("n", BATCHES)
def test_slopes_of_layers_with_fp32_results(hip, oracle, typ, n):
    import torch
    L = make_layer(typ, (64, 28, 28, 100, 3, 3, 1, 1), n, seed=9000 + n + typ)
    qw = oracle.pack_weights(L["w"], L["wthr"], weight_is_ternary(typ))
    x, thr, qw_d = (torch.from_numpy(np.ascontiguousarray(v)).cuda() for v in (L["x"], L["thr"], qw))
    for alpha in (-0.0, 0.0, 1.0, 1.5, -0.5):
        print("case", TYPE_NAMES[typ], n, alpha, flush=True)
        want = oracle.conv(typ, L["x"], L["thr"], qw, 100, 3, 3, 1, 1, alpha)
        assert (want == 0).any()
        got = hip.conv(typ, x, thr, qw_d, 100, 3, 3, 1, 1, alpha).cpu().numpy()
        assert got.tobytes() == want.tobytes(), alpha
