"""Products of operands kept in the fp4 engine's form (k_packed in fastertnn_amd/csrc/rows_kernels.hip; every form of it is reached by
tests/test_gpu_product_forms.py): tiles at ragged edges, rows shorter than a workgroup has wavefronts, K shares of every remainder, row-major and NCHW results, all
types, bit for bit against the vector-ALU engine, with nothing written past the result."""
import pytest
import torch

from fastertnn_amd import TYPE_NAMES, act_is_ternary, weight_is_ternary

pytestmark = pytest.mark.gpu

# (images, OH, OW, columns, words): tiles of 32 x 32 on four wavefronts ...
SHAPES = [(1, 1, 1, 1, 4), (33, 1, 1, 65, 4), (31, 1, 1, 32, 8), (130, 1, 1, 500, 36), (64, 1, 1, 33, 20), (2, 3, 5, 40, 12), (3, 7, 11, 129, 28),
          # ... and on eight, short and long shares
          (1, 1, 1, 1, 172), (36, 1, 1, 246, 244), (33, 1, 1, 90, 300), (1, 5, 9, 70, 204),
          # many results of short rows: tiles of 32 x 32 of the wavefronts' own; (2102, ..., 24) 64 x 32 on four wavefronts
          (645, 1, 1, 1549, 4), (3, 17, 31, 1005, 4), (2102, 1, 1, 467, 24), (1, 30, 49, 650, 24),
          # 64 x 64, 96 x 96, 128 x 128, then the wavefronts' own tiles again
          (551, 1, 1, 935, 160), (1, 20, 46, 560, 164), (1149, 1, 1, 1841, 136), (1, 43, 43, 1140, 140), (1698, 1, 1, 1874, 204), (1, 43, 44, 1700, 208),
          (1330, 1, 1, 2330, 4), (2, 32, 33, 1500, 4),
          # more than 160 tiles of 256 x 256, narrow
          (41000, 1, 1, 33, 4), (70, 1, 1, 50000, 4)]


@pytest.mark.parametrize("typ", range(4), ids=[TYPE_NAMES[t] for t in range(4)])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda v: "x".join(map(str, v)))
def test_kept_operands(hip, typ, shape):
    n, oh, ow, kn, kw = shape
    print("case", TYPE_NAMES[typ], shape, flush=True)
    g = torch.Generator(device="cuda").manual_seed(11 + typ + n + kn + kw)
    at, wt = act_is_ternary(typ), weight_is_ternary(typ)
    words = lambda rows, tern: torch.randint(-2**63, 2**63 - 1, (rows * kw * (2 if tern else 1),), generator=g, device="cuda", dtype=torch.int64)
    m, ku = n * oh * ow, 64 * kw - 7
    a, b = words(m, at), words(kn, wt)
    ea, eb = hip.expand_rows(hip.ENGINE_MFMA_F4, a, m, kw, at), hip.expand_rows(hip.ENGINE_MFMA_F4, b, kn, kw, wt)
    out = torch.full((m * kn + 64,), float("nan"), device="cuda")
    for alpha in (0.5, -0.25):
        hip.mm_expanded(hip.ENGINE_MFMA_F4, typ, ea, eb, n, oh, ow, kn, kw, alpha, ku, out=out)
        want = hip.mm_engine(hip.ENGINE_VALU, typ, a, b, n, oh, ow, kn, kw, alpha, ku).reshape(-1)
        assert torch.equal(out[:m * kn].view(torch.int32), want.view(torch.int32)), alpha
        assert bool(torch.isnan(out[m * kn:]).all())


def test_extreme_lanes(hip):
    """all lanes +1, all -1 and all 0 in rows at the length from which sums would no longer be exact, and one word"""
    for kw in (4, 65536):
        plus, minus = torch.zeros(kw, dtype=torch.int64, device="cuda"), torch.full((kw,), -1, dtype=torch.int64, device="cuda")
        a = torch.cat([plus, minus, plus])
        ea = hip.expand_rows(hip.ENGINE_MFMA_F4, a, 3, kw, False)
        got = hip.mm_expanded(hip.ENGINE_MFMA_F4, 3, ea, ea, 3, 1, 1, 3, kw, 2.0, 64 * kw).reshape(3, 3).cpu()
        L = 64.0 * kw
        assert got.tolist() == [[L, -2 * L, L], [-2 * L, L, -2 * L], [L, -2 * L, L]], kw
