"""The work that users of this library have it do, as cases that can be timed and compared.

Kinds of cases, all through the public entry points of `fastertnn_amd.lib`:

  gemm   a product of packed operands, whole call (mm_engine, engine AUTO), operands and result on the GPU
  kept   the same with both operands brought into the engine's form beforehand (expand_rows, mm_expanded)
  conv   one conv or fully connected layer with its weights prepared once (conv_prepared), tensors on the GPU
  net    a whole network as a chain of layers (Net.run), tensors on the GPU
  host   one layer through the reference's own entry point tnns_conv, tensors in host memory

Every result is an integer sum, times a slope of 0.5 where it is negative, in fp32: exact.
"""
import math

import numpy as np
import torch

import fastertnn_amd.lib as lib
from fastertnn_amd import BNN, TYPE_NAMES, act_is_ternary, shapes, weight_is_ternary

TYPES = {name: t for t, name in TYPE_NAMES.items()}
ALPHA = 0.5   # the slope of the reference's drivers

# network tables whose layers follow each other shape by shape
NETS = {"resnet18-like": [tuple(r) for r in shapes.RESNET18_LIKE]}
for _table in shapes.reference_tables()["e2e"]:
    NETS.setdefault(_table["name"], [tuple(r) for r in _table["layers"]])
CHAINED = ("resnet18-like", "resnet18", "darknet19", "darknet53", "resnet152")


def _gemm(kind, typ, m, n, p):
    return {"kind": kind, "type": typ, "m": m, "n": n, "p": p}


def _layer(kind, typ, batch, c, h, w, kn, kh, kw, pad, stride):
    return {"kind": kind, "type": typ, "batch": batch, "c": c, "h": h, "w": w, "kn": kn, "kh": kh, "kw": kw,
            "pad": pad, "stride": stride}


def listed():
    return [
        # the reference's CPU-sized GEMM: one short call, where latency and launches count
        dict(_gemm("gemm", "tnn", 256, 256, 4096), name="gemm_256"),
        # the middle of the reference's GEMM sweep (m = n, p = 8 m)
        dict(_gemm("gemm", "tnn", 1024, 1024, 8192), name="gemm_1024"),
        # a ragged product with one binary operand, as a fully connected layer over a batch of feature vectors has it
        dict(_gemm("gemm", "btn", 1999, 1733, 14592), name="gemm_ragged"),
        # the large compute-bound GEMM of the baseline
        dict(_gemm("gemm", "tnn", 8192, 8192, 32768), name="gemm_8192"),
        # the top of the reference's GEMM sweep with weights and activations kept in engine form
        dict(_gemm("kept", "tnn", 4096, 4096, 32768), name="kept_4096"),
        # single-image inference: one 3x3 layer of a mid-network stage
        dict(_layer("conv", "tnn", 1, 256, 56, 56, 256, 3, 3, 1, 1), name="conv_image"),
        # a small batch with binary weights
        dict(_layer("conv", "tbn", 8, 128, 28, 28, 128, 3, 3, 1, 1), name="conv_batch8"),
        # the largest single layer of the reference's driver at its batch of 8
        dict(_layer("conv", "tnn", 8, 1024, 56, 56, 1024, 3, 3, 1, 2), name="conv_wide"),
        # the largest fully connected layer of the reference's driver at its batch of 8
        dict(_layer("conv", "tnn", 8, 16384, 1, 1, 16384, 1, 1, 0, 1), name="fc_16384"),
        # the baseline's network, end to end on images of 224 x 224 at its batch of 32
        {"kind": "net", "net": "resnet18-like", "type": "tnn", "batch": 32, "name": "net_batch32"},
        # the deepest network of the reference's driver at its batch of 8
        {"kind": "net", "net": "resnet152", "type": "tnn", "batch": 8, "name": "net_deep"},
        # the reference's own call from C or Python programs that keep their tensors in host memory
        dict(_layer("host", "btn", 8, 128, 28, 28, 128, 3, 3, 1, 1), name="host_layer"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_layer(rng, kind, most_macs, most_values):
    while True:
        k = rng.choice((1, 1, 3, 3, 3, 5, 7))
        kw = k if rng.random() < 0.9 else rng.choice((1, 3, 5))
        h = _log(rng, 1 if k == 1 else 7, 112)
        w = h if rng.random() < 0.7 else _log(rng, max(kw, 4), 112)
        c = rng.choice((64, 128, 256, 512, 1024, _log(rng, 3, 1500), _log(rng, 3, 1500)))
        kn = rng.choice((64, 128, 256, 512, 1000, _log(rng, 10, 1500)))
        case = _layer(kind, rng.choice(sorted(TYPES)), _log(rng, 1, 64), c, h, w, kn, k, kw, rng.choice((0, k // 2, k // 2)),
                      rng.choice((1, 1, 2)))
        oh, ow = _out_dims(case)
        if oh <= 0 or ow <= 0:
            continue
        values = case["batch"] * max(c * h * w, kn * oh * ow)
        if values <= most_values and values + kn * c * k * kw >= 20000 and work(case)["flops"] <= 2 * most_macs:
            return case


def draw(rng):
    kind = rng.choice(("gemm", "gemm", "gemm", "kept", "conv", "conv", "conv", "fc", "net", "host"))
    typ = rng.choice(sorted(TYPES))
    if kind in ("gemm", "kept"):
        # from the reference sweep's smallest to the baseline's largest, square and not, p a multiple of 256
        return _gemm(kind, typ, _log(rng, 32, 8192), _log(rng, 32, 8192), 256 * _log(rng, 1, 128))
    if kind == "fc":
        return _layer("conv", typ, _log(rng, 1, 64), _log(rng, 512, 16384), 1, 1, _log(rng, 100, 16384), 1, 1, 0, 1)
    if kind == "net":
        return {"kind": "net", "net": rng.choice(CHAINED[:3]), "type": typ, "batch": _log(rng, 1, 64)}
    if kind == "conv":
        return _draw_layer(rng, "conv", 6e10, 3e7)
    return _draw_layer(rng, "host", 4e9, 1.6e6)


def _out_dims(c):
    return ((c["h"] + 2 * c["pad"] - c["kh"]) // c["stride"] + 1, (c["w"] + 2 * c["pad"] - c["kw"]) // c["stride"] + 1)


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _lanes(g, shape, ternary):
    """uniform {-1, 0, +1} or {-1, +1} as fp32"""
    if ternary:
        return torch.randint(-1, 2, shape, generator=g, device="cuda", dtype=torch.int8).float()
    return torch.randint(0, 2, shape, generator=g, device="cuda", dtype=torch.int8).float() * 2 - 1


def _operand(g, rows, p, ternary):
    """packed rows of a GEMM operand with uniform lanes"""
    if not ternary:
        return torch.randint(-2**63, 2**63 - 1, (rows * p // 64,), generator=g, device="cuda", dtype=torch.int64)
    return lib.pack_gemm_operand(_lanes(g, (rows, p), True))


def _packed_weights(g, kn, c, kh, kw, typ):
    wt = weight_is_ternary(typ)
    return lib.pack_weights(_lanes(g, (kn, c, kh, kw), wt), torch.full((kn,), 0.5 if wt else 0.0, device="cuda"), wt)


def prepare(case, seed):
    g = _generator(seed)
    s = dict(case)
    kind, typ = case["kind"], TYPES[case["type"]]
    s["t"] = typ
    at = act_is_ternary(typ)
    thr = 0.5 if at else 0.0   # the baseline's thresholds for N(0, 1) inputs
    if kind in ("gemm", "kept"):
        m, n, k = case["m"], case["n"], case["p"] // 64
        a, b = _operand(g, m, case["p"], at), _operand(g, n, case["p"], weight_is_ternary(typ))
        s["k"], s["k_unpack"] = k, case["p"] if typ == BNN else 0
        s["out"] = torch.empty((m, n, 1, 1), device="cuda")
        if kind == "gemm":
            need = lib.mm_scratch_bytes(lib.ENGINE_AUTO, typ, m, 1, 1, n, k)
            s["a"], s["b"], s["scratch"] = a, b, torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
        else:
            s["a"] = lib.expand_rows(lib.ENGINE_MFMA_F4, a, m, k, at)
            s["b"] = lib.expand_rows(lib.ENGINE_MFMA_F4, b, n, k, weight_is_ternary(typ))
        return s
    n = case["batch"]
    if kind == "net":
        table = NETS[case["net"]]
        layers = [dict(type=typ, shape=row, threshold=thr, alpha=ALPHA,
                       qw=_packed_weights(g, row[3], row[0], row[5], row[4], typ)) for row in table]
        s["net"] = lib.Net(n, layers)
        s["x"] = torch.randn((n,) + table[0][:3], generator=g, device="cuda")
        s["out"] = torch.empty(s["net"].out_shape, device="cuda")
        return s
    c, h, w, kn, kh, kw, pad, stride = (case[v] for v in ("c", "h", "w", "kn", "kh", "kw", "pad", "stride"))
    oh, ow = _out_dims(case)
    x = torch.randn((n, c, h, w), generator=g, device="cuda")
    qw = _packed_weights(g, kn, c, kh, kw, typ)
    if kind == "host":
        s["x"], s["thr"], s["qw"] = x.cpu().numpy(), np.full(n, thr, np.float32), qw.cpu().numpy()
        return s
    s["x"], s["thr"] = x, torch.full((n,), thr, device="cuda")
    s["w"] = lib.prepare_conv_weights(typ, qw, c, kn, kh, kw)
    s["scratch"] = torch.empty(lib.conv_scratch_bytes(typ, n, c, h, w, kn, kh, kw, pad, stride), dtype=torch.uint8,
                               device="cuda")
    s["out"] = torch.empty((n, kn, oh, ow), device="cuda")
    return s


def run(s):
    kind, t = s["kind"], s["t"]
    if kind == "gemm":
        return lib.mm_engine(lib.ENGINE_AUTO, t, s["a"], s["b"], s["m"], 1, 1, s["n"], s["k"], ALPHA,
                             k_unpack=s["k_unpack"], out=s["out"], scratch=s["scratch"])
    if kind == "kept":
        return lib.mm_expanded(lib.ENGINE_MFMA_F4, t, s["a"], s["b"], s["m"], 1, 1, s["n"], s["k"], ALPHA,
                               k_unpack=s["k_unpack"], out=s["out"])
    if kind == "net":
        return s["net"].run(s["x"], out=s["out"])
    if kind == "host":
        return lib.host_conv(t, s["x"], s["thr"], s["qw"], s["kn"], s["kh"], s["kw"], s["pad"], s["stride"], ALPHA)
    return lib.conv_prepared(t, s["x"], s["thr"], s["w"], s["kn"], s["kh"], s["kw"], s["pad"], s["stride"], ALPHA,
                             scratch=s["scratch"], out=s["out"])


def work(case):
    """inputs once and outputs once; weights and packed operands at the bits of their Packing-2 rows"""
    kind, typ = case["kind"], TYPES[case["type"]]
    abits, wbits = (2 if act_is_ternary(typ) else 1), (2 if weight_is_ternary(typ) else 1)
    if kind in ("gemm", "kept"):
        m, n, p = case["m"], case["n"], case["p"]
        return {"bytes": (m * abits + n * wbits) * p / 8 + 4 * m * n, "flops": 2 * m * n * p}
    b = case["batch"]
    if kind == "net":
        rows = NETS[case["net"]]
        c, h, w = rows[0][:3]
        oh = (rows[-1][1] + 2 * rows[-1][6] - rows[-1][5]) // rows[-1][7] + 1
        ow = (rows[-1][2] + 2 * rows[-1][6] - rows[-1][4]) // rows[-1][7] + 1
        weights = sum(r[0] * r[3] * r[4] * r[5] for r in rows) * wbits / 8
        return {"bytes": 4 * b * (c * h * w + rows[-1][3] * oh * ow) + weights,
                "flops": 2 * sum(shapes.layer_macs(b, r) for r in rows)}
    oh, ow = _out_dims(case)
    k = case["c"] * case["kh"] * case["kw"]
    values_in = 4 * b * case["c"] * case["h"] * case["w"]
    return {"bytes": values_in + 4 * b * case["kn"] * oh * ow + case["kn"] * k * wbits / 8,
            "flops": 2 * b * oh * ow * case["kn"] * k}


def tolerance(case):
    return "exact"
