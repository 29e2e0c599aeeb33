"""Products on wavefronts with tiles of their own and on eight that split K, and results stored through the caches (k_rows and k_packed
in fastertnn_amd/csrc/rows_kernels.hip): tiles with one row or column inside, wavefronts whose tile lies outside the product, shares of K of
every remainder, row-major and NCHW results, all types, bit for bit against the vector-ALU engine, with nothing written past the
result."""
import pytest
import torch

from fastertnn_amd import TYPE_NAMES, act_is_ternary, weight_is_ternary

pytestmark = pytest.mark.gpu

# (images, OH, OW, columns, words): mostly a tile per wavefront, rows of one to seven groups; 33 and 97 leave one row or column to a
# workgroup's second wavefronts or none, 1025 to the first ones
SHAPES = [(33, 1, 1, 20000, 4), (20000, 1, 1, 33, 8), (1025, 1, 1, 897, 4), (897, 1, 1, 1025, 12), (2, 23, 31, 961, 16), (97, 7, 97, 65, 4), (1, 1, 700000, 1, 4),
          (700000, 1, 1, 1, 4), (1600, 1, 1, 1601, 28),
          # eight wavefronts that split K
          (1, 1, 1, 1, 128), (31, 1, 1, 97, 260), (3, 5, 7, 129, 300), (65, 1, 1, 33, 1000), (257, 1, 1, 131, 452),
          # rows that are no whole sectors of results beyond 4 Mi: through the caches, on the wavefronts' own tiles and after a meeting
          (2300, 1, 1, 2301, 4), (5, 21, 23, 2211, 8), (2297, 1, 1, 2303, 140), (5, 21, 23, 2209, 132),
          # 160 tiles of 256 x 256 and more: wavefronts on 2 x 2 blocks of their own, with one block, row or column inside, or none
          (3105, 1, 1, 3361, 32), (5, 25, 27, 3169, 28), (6177, 1, 1, 1825, 40), (41, 11, 13, 1889, 36), (3137, 1, 1, 3201, 64),
          # longer rows of such products: on the same, on four wavefronts that share a tile of 128 x 128, and both operands packed first
          (4129, 1, 1, 2593, 100), (4129, 1, 1, 2625, 260), (3, 37, 41, 2593, 100), (20001, 1, 1, 609, 128)]
# Every form of kRowsForms and kPackedForms (fastertnn_amd/csrc/product_forms.h; 7: packed first, 9: k_mfma_p4), row-major and NCHW, past and through the
# caches, ragged: (form from packed rows, form of kept operands), which tests/test_product_forms.py holds the shapes to
FORMS = {(3018, 1, 1, 1, 4): (0, 0), (4300001, 1, 1, 1, 4): (4, 7), (1, 2100, 2051, 1, 4): (4, 7), (8290, 1, 1, 38, 44): (1, 0),
         (3, 59, 22, 1098, 48): (1, 7), (26, 19, 17, 41, 40): (1, 0), (1897, 1, 1, 2399, 96): (2, 5), (19790, 1, 1, 70, 56): (2, 3),
         (2, 22, 20, 4835, 88): (2, 4), (24820, 1, 1, 237, 108): (3, 8), (29241, 1, 1, 82, 84): (6, 8), (10, 37, 67, 233, 112): (3, 8),
         (10, 49, 5, 1225, 84): (6, 8), (40004, 1, 1, 105, 4): (4, 7), (11, 15, 6, 4238, 4): (4, 7), (11, 41, 20, 52, 4): (4, 7),
         (3, 1, 1, 1057, 80): (5, 0), (25, 5, 12, 2, 80): (5, 0), (54522, 1, 1, 88, 20): (6, 8), (24, 69, 46, 71, 16): (6, 8),
         (13, 34, 57, 94, 28): (6, 8), (5100, 1, 1, 2701, 400): (7, 9), (5100, 1, 1, 2704, 400): (7, 9), (3, 41, 41, 2700, 400): (7, 9),
         (3, 40, 42, 2701, 400): (7, 9), (35, 44, 2, 1, 116): (5, 1), (1, 1, 1, 3007, 116): (5, 1), (769, 1, 1, 6430, 80): (1, 2),
         (34, 42, 12, 277, 68): (1, 2), (9342, 1, 1, 531, 88): (1, 3), (1, 2, 4, 8936, 20): (0, 3), (12897, 1, 1, 332, 76): (1, 4),
         (18, 33, 42, 179, 72): (1, 4), (3, 4, 3, 8435, 72): (1, 4), (462, 1, 1, 4678, 40): (2, 5), (2, 23, 33, 2894, 92): (2, 5),
         (12878, 1, 1, 213, 156): (3, 6), (8, 31, 43, 330, 128): (3, 6), (4129, 1, 1, 2625, 400): (3, 6), (3, 37, 37, 2601, 300): (3, 6),
         (215, 1, 1, 4267, 112): (0, 2), (1, 37, 141, 73, 252): (0, 2)}


def _products(hip, typ, shape, alpha):
    """the product by whole call and of kept operands against the vector-ALU engine, nothing written past the result"""
    n, oh, ow, kn, kw = shape
    print("case", TYPE_NAMES[typ], shape, flush=True)
    g = torch.Generator(device="cuda").manual_seed(5 + typ + n + kn + kw)
    at, wt = act_is_ternary(typ), weight_is_ternary(typ)
    words = lambda rows, tern: torch.randint(-2**63, 2**63 - 1, (rows * kw * (2 if tern else 1),), generator=g, device="cuda", dtype=torch.int64)
    m, ku = n * oh * ow, 64 * kw - 9
    a, b = words(m, at), words(kn, wt)
    ea, eb = hip.expand_rows(hip.ENGINE_MFMA_F4, a, m, kw, at), hip.expand_rows(hip.ENGINE_MFMA_F4, b, kn, kw, wt)
    want = hip.mm_engine(hip.ENGINE_VALU, typ, a, b, n, oh, ow, kn, kw, alpha, ku).reshape(-1)
    for kept in (False, True):
        out = torch.full((m * kn + 64,), float("nan"), device="cuda")
        if kept:
            hip.mm_expanded(hip.ENGINE_MFMA_F4, typ, ea, eb, n, oh, ow, kn, kw, alpha, ku, out=out)
        else:
            hip.mm_engine(hip.ENGINE_MFMA_F4, typ, a, b, n, oh, ow, kn, kw, alpha, ku, out=out)
        assert torch.equal(out[:m * kn].view(torch.int32), want.view(torch.int32)), kept
        assert bool(torch.isnan(out[m * kn:]).all())


@pytest.mark.parametrize("shape", FORMS, ids=lambda v: "x".join(map(str, v)))
def test_every_form(hip, shape):
    for typ in range(4):
        _products(hip, typ, shape, 0.5 if typ % 2 else -0.25)


@pytest.mark.parametrize("typ", range(4), ids=[TYPE_NAMES[t] for t in range(4)])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda v: "x".join(map(str, v)))
def test_product_forms(hip, typ, shape):
    _products(hip, typ, shape, -0.25)


@pytest.mark.parametrize("typ", range(4), ids=[TYPE_NAMES[t] for t in range(4)])
@pytest.mark.parametrize("shape", [(3328, 1, 1, 3328, 16), (4, 29, 29, 3200, 16)], ids=lambda v: "x".join(map(str, v)))
def test_result_over_an_operand(hip, typ, shape):
    """products of 160 tiles of 256 x 256 and more of short rows, with scratch, the result from an operand's first and last word on: as in a place of its own"""
    n, oh, ow, kn, kw = shape
    print("case", TYPE_NAMES[typ], shape, flush=True)
    g = torch.Generator(device="cuda").manual_seed(8 + typ)
    at, wt = act_is_ternary(typ), weight_is_ternary(typ)
    words = lambda rows, tern: torch.randint(-2**63, 2**63 - 1, (rows * kw * (2 if tern else 1),), generator=g, device="cuda", dtype=torch.int64)
    m = n * oh * ow
    a, b = words(m, at), words(kn, wt)
    scratch = torch.empty(hip.mm_scratch_bytes(hip.ENGINE_AUTO, typ, n, oh, ow, kn, kw), dtype=torch.uint8, device="cuda")
    want = hip.mm_engine(hip.ENGINE_VALU, typ, a, b, n, oh, ow, kn, kw, 0.5, 64 * kw - 9)
    for engine in (hip.ENGINE_AUTO, hip.ENGINE_MFMA_F4):
        for which in (0, 1):
            for at_end in (False, True):
                own, other = (a, b) if which == 0 else (b, a)
                buf = torch.empty(own.numel() + (m * kn + 1) // 2, dtype=torch.int64, device="cuda")
                held = buf[:own.numel()]
                held.copy_(own)
                start = 2 * (own.numel() - 1) if at_end else 0
                out = buf.view(torch.float32)[start:start + m * kn].view(n, kn, oh, ow)
                hip.mm_engine(engine, typ, *((held, other) if which == 0 else (other, held)), n, oh, ow, kn, kw, 0.5, 64 * kw - 9, out=out, scratch=scratch)
                assert torch.equal(out, want), (engine, which, at_end)
