"""The matrix-core GEMM straight from packed rows (k_rows, what the explicit fp4 engine runs below 160 tiles of 256 x 256, and AUTO
where the vector ALU is not ahead): every type, row-major and NCHW results, at the sizes where each of its wavefront
tiles starts, ends or is ragged, with K from one group of words (fewer groups than wavefronts) to K tails, bit for bit
against the oracle."""
import numpy as np
import pytest

from fastertnn_amd import BNN, TNN, TYPE_NAMES, act_is_ternary, weight_is_ternary
from tests.cases import ALL_TYPES

pytestmark = pytest.mark.gpu

# (n, oh, ow, kn, words): by the launcher's estimates on tiles of 32 x 32 up to the single row and the narrow products,
# then 64 x 64, 96 x 96 and 128 x 128
SHAPES = [(1, 1, 1, 1, 4), (32, 1, 1, 32, 4), (33, 1, 1, 65, 8), (3, 5, 7, 31, 12), (2, 16, 16, 96, 20), (8, 1, 1, 1000, 64),
          (1000, 1, 1, 7, 4), (129, 1, 1, 257, 36), (897, 1, 1, 900, 128), (5, 13, 14, 901, 132), (1300, 1, 1, 1299, 160),
          (9, 12, 12, 1310, 160), (1999, 1, 1, 1733, 68), (2, 31, 31, 2050, 64)]


def _operands(typ, m, kn, kw, seed):
    rng = np.random.default_rng(seed)
    at, wt = act_is_ternary(typ), weight_is_ternary(typ)
    return (rng.integers(-2 ** 63, 2 ** 63, size=m * kw * (2 if at else 1), dtype=np.int64),
            rng.integers(-2 ** 63, 2 ** 63, size=kn * kw * (2 if wt else 1), dtype=np.int64))


@pytest.mark.parametrize("typ", ALL_TYPES, ids=lambda t: TYPE_NAMES[t])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_products_from_packed_rows(hip, oracle, typ, shape):
    import torch
    n, oh, ow, kn, kw = shape
    m = n * oh * ow
    print("case", TYPE_NAMES[typ], shape, flush=True)
    a, b = _operands(typ, m, kn, kw, 100 * typ + m + kn + kw)
    ku = 64 * kw - 5
    a_d, b_d = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()
    for alpha in (0.5, -0.25):
        want = oracle.mm(typ, a, b, n, oh, ow, kn, kw, alpha, ku)
        for engine in (hip.ENGINE_MFMA_F4, hip.ENGINE_AUTO):
            # a sentinel past the result: nothing may be written there
            y = torch.full((m * kn + 64,), float("nan"), dtype=torch.float32, device="cuda")
            hip.mm_engine(engine, typ, a_d, b_d, n, oh, ow, kn, kw, alpha, ku, out=y)
            got = y.cpu().numpy()
            assert got[:m * kn].tobytes() == want.tobytes(), (engine, alpha)
            assert np.isnan(got[m * kn:]).all()


def test_rows_longer_than_the_fp4_engine_takes(hip):
    """AUTO runs rows beyond the packed4 form's 65536 words from the packed rows too, up to 2^18 words: lanes almost all
    +1 on both sides, sums near 2^23, against the vector ALU's integers"""
    import torch
    rng = np.random.default_rng(5)
    m, n, kw = 3, 5, (1 << 17) + 4
    r = rng.integers(-2 ** 63, 2 ** 63, size=(5, (m + n) * 2 * kw), dtype=np.int64)
    rows = r[0] & r[1] & r[2] & r[3] & r[4]
    d = torch.from_numpy(rows).cuda()
    a_d, b_d = d[:m * 2 * kw].contiguous(), d[m * 2 * kw:].contiguous()
    print("case long rows", m, n, kw, flush=True)
    want = hip.mm_engine(hip.ENGINE_VALU, TNN, a_d, b_d, m, 1, 1, n, kw, 0.5).cpu().numpy()
    got = hip.mm_engine(hip.ENGINE_AUTO, TNN, a_d, b_d, m, 1, 1, n, kw, 0.5).cpu().numpy()
    assert want.max() > 6_000_000 and got.tobytes() == want.tobytes()


def test_large_product_without_scratch(hip, oracle):
    """a product of 160 tiles of 256 x 256 and more whose caller brings no scratch"""
    import torch
    m, n, kw = 3333, 3100, 4
    a, b = _operands(TNN, m, n, kw, 9)
    want = oracle.mm(TNN, a, b, m, 1, 1, n, kw, 0.5)
    y = torch.empty(m * n, device="cuda")
    a_d, b_d = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()
    rc = hip._L.ftnn_mm_engine(hip.ENGINE_AUTO, TNN, a_d.data_ptr(), b_d.data_ptr(), m, 1, 1, n, kw, 0, 0.5, y.data_ptr(), None, 0,
                               hip._stream())
    assert rc == 0 and y.cpu().numpy().tobytes() == want.tobytes()


def test_more_rows_than_the_smallest_tile_has_workgroups_for(hip):
    """one column under 2^29 + 33 rows: 2^24 + 2 tiles of 32 x 32 would be 2^32 threads and more, which no launch takes; the
    next larger tile does it, against the vector ALU's integers"""
    import torch
    m, kw = (1 << 29) + 33, 4
    print("case many rows", m, kw, flush=True)
    torch.manual_seed(3)
    a_d = torch.randint(-2 ** 62, 2 ** 62, (m * kw,), dtype=torch.int64, device="cuda")
    b_d = torch.randint(-2 ** 62, 2 ** 62, (kw,), dtype=torch.int64, device="cuda")
    want = hip.mm_engine(hip.ENGINE_VALU, BNN, a_d, b_d, m, 1, 1, 1, kw, 0.5, 64 * kw)
    got = hip.mm_engine(hip.ENGINE_MFMA_F4, BNN, a_d, b_d, m, 1, 1, 1, kw, 0.5, 64 * kw)
    assert torch.equal(got, want)


@pytest.mark.parametrize("typ", ALL_TYPES, ids=lambda t: TYPE_NAMES[t])
@pytest.mark.parametrize("shape", [(41000, 99, 8), (99, 41000, 8)], ids=["narrow", "low"])
def test_explicit_fp4_engine_on_narrow_products(hip, oracle, typ, shape):
    """products of 160 tiles of 256 x 256 and more that are narrower than 128 run from the packed rows on the explicit engine too,
    with scratch for both operands in packed4 form, which stays as it was; less is refused"""
    import torch
    m, n, kw = shape
    a, b = _operands(typ, m, n, kw, 7 + typ)
    ku = 64 * kw - 9
    print("case", TYPE_NAMES[typ], shape, flush=True)
    want = oracle.mm(typ, a, b, m, 1, 1, n, kw, 0.5, ku)
    a_d, b_d = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()
    packed4 = sum(int(hip._L.ftnn_expand_bytes(hip.ENGINE_MFMA_F4, r, kw)) for r in (m, n))
    assert hip.mm_scratch_bytes(hip.ENGINE_MFMA_F4, typ, m, 1, 1, n, kw) == packed4
    scratch = torch.full((packed4,), 0x5A, dtype=torch.uint8, device="cuda")
    got = hip.mm_engine(hip.ENGINE_MFMA_F4, typ, a_d, b_d, m, 1, 1, n, kw, 0.5, ku, scratch=scratch).cpu().numpy()
    assert got.tobytes() == want.tobytes()
    assert bool((scratch == 0x5A).all())
    with pytest.raises(hip.FtnnError):
        hip.mm_engine(hip.ENGINE_MFMA_F4, typ, a_d, b_d, m, 1, 1, n, kw, 0.5, ku, scratch=scratch[:packed4 - 1].contiguous())
