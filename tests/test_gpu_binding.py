"""The calls that go through csrc/py_call.cpp: what it reads itself gives the results of the way through ctypes, and what it
leaves to that way is still converted, refused or reported as there."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")
import fastertnn_amd.lib as lib
from fastertnn_amd import BTN, TNN

pytestmark = pytest.mark.gpu


class _NoCall:
    """every function leaves its call to ctypes"""

    def __getattr__(self, name):
        return lambda *args: None


def _calls():
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    words = lambda n: torch.randint(-2**63, 2**63 - 1, (n,), generator=g, device="cuda", dtype=torch.int64)
    m, n, k = 70, 130, 8
    a, b = words(m * 2 * k), words(n * 2 * k)
    scratch = torch.empty(1 << 20, dtype=torch.uint8, device="cuda")
    ea, eb = (lib.expand_rows(lib.ENGINE_MFMA_F4, t, r, k, True) for t, r in ((a, m), (b, n)))
    x = torch.randn((2, 96, 9, 7), generator=g, device="cuda")
    thr = torch.full((2,), 0.5, device="cuda")
    qw = words(40 * lib.row_words(96, 3, 3, True))
    prep = lib.prepare_conv_weights(TNN, qw, 96, 40, 3, 3)
    y = lambda *s: torch.full(s, 7.0, device="cuda")
    layer = (3, 3, 1, 2, 0.25)   # kh, kw, pad, stride, alpha
    net = lib.Net(2, [dict(type=TNN, shape=(96, 9, 7, 40, 3, 3, 1, 2), threshold=0.5, alpha=0.25, qw=qw)])
    return {
        "mm": lambda: lib.mm(TNN, a, b, m, 1, 1, n, k, 0.25, out=y(m, n, 1, 1)),
        "mm_engine": lambda: lib.mm_engine(lib.ENGINE_AUTO, TNN, a, b, m, 1, 1, n, k, 0.25, out=y(m, n, 1, 1), scratch=scratch),
        "mm_expanded": lambda: lib.mm_expanded(lib.ENGINE_MFMA_F4, TNN, ea, eb, m, 1, 1, n, k, 0.25, out=y(m, n, 1, 1)),
        "conv": lambda: lib.conv(TNN, x, thr, qw, 40, *layer, scratch=scratch, out=y(2, 40, 5, 4)),
        "conv_prepared": lambda: lib.conv_prepared(TNN, x, thr, prep, 40, *layer, scratch=scratch, out=y(2, 40, 5, 4)),
        "conv_static": lambda: lib.conv_static(TNN, x, thr, qw, 40, *layer, y(2, 40, 5, 4)),
        "net_run": lambda: net.run(x, out=y(2, 40, 5, 4)),
    }


def test_same_results_as_through_ctypes(monkeypatch):
    calls = _calls()
    native, answered = lib._native(), []

    class Spy:
        def __getattr__(self, name):
            def fn(*args):
                rc = getattr(native, name)(*args)
                answered.append((name, rc))
                return rc
            return fn

    monkeypatch.setattr(lib, "_call", Spy())
    fast = {n: f().cpu() for n, f in calls.items()}
    assert answered == [(n, 0) for n in calls]   # each was taken, and none refused
    monkeypatch.setattr(lib, "_call", _NoCall())
    for n, f in calls.items():
        assert torch.equal(fast[n], f().cpu()), n


def test_arguments_it_does_not_read_itself():
    """numpy integers, an integer slope, no output, no scratch: through ctypes, same results"""
    g = torch.Generator(device="cuda")
    g.manual_seed(6)
    a, b = (torch.randint(-2**63, 2**63 - 1, (r * 8,), generator=g, device="cuda", dtype=torch.int64) for r in (33, 65))
    out = lambda: torch.empty((33, 65, 1, 1), device="cuda")
    want = lib.mm(TNN, a, b, 33, 1, 1, 65, 4, 1.0, out=out())
    assert torch.equal(want, lib.mm(TNN, a, b, np.int64(33), 1, 1, np.int32(65), 4, 1, out=out()))
    assert torch.equal(want, lib.mm(TNN, a, b, 33, 1, 1, 65, 4, 1.0))
    assert torch.equal(want, lib.mm_engine(lib.ENGINE_AUTO, TNN, a, b, 33, 1, 1, 65, 4, 1.0))
    sub = a.as_subclass(type("Sub", (torch.Tensor,), {}))
    assert torch.equal(want, lib.mm(TNN, sub, b, 33, 1, 1, 65, 4, 1.0, out=out()))


def test_what_is_refused():
    g = torch.zeros(33 * 8, dtype=torch.int64, device="cuda")
    out = torch.empty((33, 33, 1, 1), device="cuda")
    mm = lambda a, b, out: lib.mm(TNN, a, b, 33, 1, 1, 33, 4, 0.5, out=out)
    with pytest.raises(AssertionError, match="contiguous CUDA"):
        mm(g.cpu(), g, out)
    with pytest.raises(AssertionError, match="contiguous CUDA"):
        mm(torch.zeros((4, 66), dtype=torch.int64, device="cuda").t(), g, out)
    with pytest.raises(AssertionError, match="float32"):
        mm(g, g, out.half())
    with pytest.raises(lib.FtnnError, match="ftnn error -1"):
        lib.mm(9, g, g, 33, 1, 1, 33, 4, 0.5, out=out)
    with pytest.raises(lib.FtnnError):
        lib.mm(BTN, g, g, 33, 1, 1, 0, 4, 0.5, out=out)
    with pytest.raises(ctypes.ArgumentError):
        lib.mm(TNN, g, g, "33", 1, 1, 33, 4, 0.5, out=out)


def test_runs_on_the_current_stream():
    """inputs made on a stream of its own, used on the same one with no wait of the host's"""
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        a = torch.zeros(256 * 8, dtype=torch.int64, device="cuda")
        for _ in range(50):
            a.add_(1)
        a.fill_(-1)
        out = lib.mm(3, a[:1024], a[1024:], 256, 1, 1, 256, 4, 1.0, k_unpack=256, out=torch.empty((256, 256, 1, 1), device="cuda"))
    s.synchronize()
    assert bool((out == 256).all())
