"""Tile kernels on results above and below 4 Mi values whose rows are and are not whole 64-byte sectors: the two ways their
results leave, against the exact product of the decoded lanes."""
import pytest
import torch

from fastertnn_amd import BNN, BTN, TBN, TNN, act_is_ternary, weight_is_ternary

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("typ", [TNN, TBN, BTN, BNN])
@pytest.mark.parametrize("engine,kept", [("f4", False), ("f4", True), ("i8", True)])
@pytest.mark.parametrize("m,n", [(4099, 1031), (4099, 1040), (16400, 257), (1031, 4067), (4096, 1024)])
def test_result_rows(hip, typ, engine, kept, m, n):
    eng, p, alpha = {"f4": hip.ENGINE_MFMA_F4, "i8": hip.ENGINE_MFMA_I8}[engine], 256, 0.25
    g = torch.Generator(device="cuda").manual_seed(m + n)

    def operand(rows, ternary):
        if ternary:
            x = torch.randint(-1, 2, (rows, p), generator=g, device="cuda").float()
            return x, hip.pack_gemm_operand(x)
        x = torch.randint(0, 2, (rows, p), generator=g, device="cuda").float() * 2 - 1
        bits = (x < 0).long().view(rows, p // 64, 64) << torch.arange(64, device="cuda")
        return x, bits.sum(-1).reshape(-1)

    a, ap = operand(m, act_is_ternary(typ))
    b, bp = operand(n, weight_is_ternary(typ))
    want = (a.cpu() @ b.cpu().T).double()
    want = torch.where(want < 0, want * alpha, want).float()
    args = (eng, typ)
    tail = (m, 1, 1, n, p // 64, alpha)
    ku = p if typ == BNN else 0
    out = torch.full((m, n, 1, 1), float("nan"), device="cuda")
    if kept:
        ax, bx = hip.expand_rows(eng, ap, m, p // 64, act_is_ternary(typ)), hip.expand_rows(eng, bp, n, p // 64, weight_is_ternary(typ))
        got = hip.mm_expanded(*args, ax, bx, *tail, k_unpack=ku, out=out)
    else:
        got = hip.mm_engine(*args, ap, bp, *tail, k_unpack=ku, out=out)
    assert torch.equal(got.view(m, n).cpu(), want)   # integer sums below 2^9, quarters: exact
