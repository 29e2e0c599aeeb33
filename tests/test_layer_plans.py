"""The rules by which layers are cut into launches (fastertnn_amd/csrc/layer_plans.h, the code the launchers run): the grid over the dense
rows of a few-channel layer, up to the most output pixels a call may have, which form makes them and where few kernels leave the matrix cores, the
comparison of a result's place with its input's, which layers run in one launch, and how the layer kernel cuts the others.  CPU only."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _run(tmp_path, program):
    src, exe = tmp_path / "plans.cpp", tmp_path / "plans"
    src.write_text('#include <stdio.h>\n#include <stdlib.h>\n#include "layer_plans.h"\nusing namespace ftnn;\n' + program)
    subprocess.run(["g++", "-O1", "-std=c++17", "-fsanitize=undefined", "-fno-sanitize-recover=all", "-I", os.path.join(ROOT, "fastertnn_amd", "csrc"),
                    str(src), "-o", str(exe)], check=True, timeout=120)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-500:] + r.stderr[-500:]
    return r.stdout


def test_grid_of_dense_rows(tmp_path):
    """every block of 32 rows once, no dimension beyond a launch's, no row index beyond 32 bits"""
    out = _run(tmp_path, r"""
int main() {
    const long long M[] = {1, 32, 33, 65535, 65536, (1LL << 28) - 31, 1LL << 28, (1LL << 28) + 1, (1LL << 29) - 32, (1LL << 29) - 31, 1LL << 29, 1LL << 30, (1LL << 30) + 1, 0x7fffffffLL};
    for (long long m : M)
        for (int groups : {1, 3, 65535, 65536, 1 << 20}) {
            const DenseGrid g = dense_rows_grid(m, groups);
            const long long blocks = (m + 31) / 32, last = (long long)(g.z - 1) * kDenseBlocksX + g.x - 1;
            if (g.x * 256LL >= 1LL << 32 || g.y < 1 || g.y > 65535 || g.z < 1 || g.z > 65535 || (long long)g.y > groups) return printf("%lld: grid\n", m), 1;
            if (g.x > kDenseBlocksX || (g.z > 1 && g.x != kDenseBlocksX) || last < blocks - 1 || (g.z > 1 && (g.z - 1) * (long long)kDenseBlocksX >= blocks)) return printf("%lld: blocks\n", m), 1;
            if (last * 32 + 31 >= 1LL << 32) return printf("%lld: rows\n", m), 1;
        }
    printf("ok\n");
}
""")
    assert out == "ok\n"


def test_ranges_that_meet(tmp_path):
    out = _run(tmp_path, r"""
int main() {
    const char* p = (const char*)0x7f0000001000ull;
    struct { long a, an, b, bn; bool meet; } c[] = {{0, 64, 64, 64, 0}, {64, 64, 0, 64, 0}, {0, 64, 63, 1, 1}, {63, 1, 0, 64, 1}, {0, 64, 0, 64, 1}, {16, 4, 0, 64, 1},
                                                    {0, 64, 16, 4, 1}, {0, 1L << 40, (1L << 40) - 4, 4, 1}, {0, 1L << 40, 1L << 40, 4, 0}};
    for (auto& v : c)
        if (ranges_meet(p + v.a, v.an, p + v.b, v.bn) != v.meet) return printf("%ld %ld\n", v.a, v.b), 1;
    printf("ok\n");
}
""")
    assert out == "ok\n"


def test_form_of_dense_rows(tmp_path):
    """sides of the line that were measured more than a tenth apart, and inputs that 32-bit offsets do not reach"""
    from tests.test_gpu_few_channels import FEW_PLANES, PLANES
    planes = ""
    for n, c, h, w, kn, kh, kw, pad, stride in PLANES + FEW_PLANES:
        oh, ow = (h + 2 * pad - kh) // stride + 1, (w + 2 * pad - kw) // stride + 1
        planes += "{0, %d, %d, %d, %d, %d, %d, 0}, {1, %d, %d, %d, %d, %d, %d, 0}, " % (2 * (n, c, h * w, oh * ow, kh * kw, stride))
    out = _run(tmp_path, r"""
int main() {
    struct { bool tern; long n; int c, hw, oh, taps, stride; bool input; } v[] = {
        {0, 22, 9, 209 * 209, 207 * 207, 9, 1, 1}, {1, 52, 11, 45 * 45, 53 * 45, 9, 1, 1}, {1, 11, 16, 15 * 16, 15 * 16, 9, 1, 1}, {1, 64, 16, 56 * 56, 56 * 56, 9, 1, 1},
        {0, 61, 19, 186 * 186, 89 * 89, 81, 2, 0}, {1, 26, 17, 70 * 70, 30 * 30, 121, 2, 0}, {0, 60, 14, 223 * 18, 207 * 2, 289, 1, 0}, {1, 42, 12, 206 * 206, 196 * 196, 121, 1, 0},
        {0, 26, 17, 63 * 63, 27 * 27, 121, 2, 0}, {1, 36, 16, 211 * 48, 211 * 48, 25, 1, 0},
        {1, 16383, 16, 64 * 64, 1, 9, 64, 1}, {1, 16384, 16, 64 * 64, 1, 9, 64, 0}, """ + planes + r"""};
    for (auto& l : v)
        if (dense_rows_from_input(l.tern, l.n * l.hw, l.c, l.n * l.oh, l.taps, l.stride) != l.input) return printf("%ld x %d, %d taps\n", l.n, l.c, l.taps), 1;
    printf("ok\n");
}
""")
    assert out == "ok\n"


def test_few_kernels(tmp_path):
    """layers of few kernels that measured slower off the vector ALU, and neighbours that measured faster"""
    out = _run(tmp_path, r"""
int main() {
    struct { long m; int kn, kw; bool valu; } v[] = {{65536, 8, 4, 1}, {61852, 8, 8, 1}, {57024, 3, 28, 1}, {89787, 1, 20, 1}, {28611, 6, 36, 1}, {56295, 1, 44, 1},
                                                    {212064, 3, 32, 0}, {119070, 3, 44, 0}, {13482, 6, 60, 0}, {10000, 10, 60, 0}, {153164, 12, 12, 0}, {65536, 16, 4, 0}};
    for (auto& l : v)
        if (few_kernels(l.m, l.kn, l.kw) != l.valu) return printf("%ld %d %d\n", l.m, l.kn, l.kw), 1;
    printf("ok\n");
}
""")
    assert out == "ok\n"


def _plans(tmp_path, layers):
    """of each layer and type: whether it runs in one launch, lgS, workgroups per tile"""
    geoms = []
    for n, c, h, w, kn, kh, kw, pad, stride in layers:
        oh, ow = (h + 2 * pad - kh) // stride + 1, (w + 2 * pad - kw) // stride + 1
        geoms.append("{%d, %d, %d, %d, %d, %d, %d, %d, %d, %d, %d}" % (n, c, h, w, kn, kh, kw, pad, stride, oh, ow))
    out = _run(tmp_path, r"""
int main() {
    const int layers[][11] = {""" + ", ".join(geoms) + r"""};
    for (auto& l : layers) {
        const int cp = cpack_of(l[1]);
        const ConvGeom cg = {l[2], l[3], cp, l[9], l[10], l[6], cp * l[5] * l[6], l[7], l[7], l[8], l[8], make_fastdiv((uint32_t)l[10]), make_fastdiv((uint32_t)cp), make_fastdiv((uint32_t)l[6])};
        for (int type = 0; type < 4; type++) {
            DirectPlan p;
            const bool runs = direct_plan(type, cg, l[1], l[0], l[4], &p);
            if (runs && (p.lds_bytes > 65536 || p.tiles * p.groups > 400 || (p.groups << (3 - p.lgS)) * 32 < l[4])) exit(1);
            printf("%d %d %d\n", runs, p.lgS, p.groups);
        }
    }
}
""").split()
    v = [(out[i] == "1", int(out[i + 1]), int(out[i + 2])) for i in range(0, len(out), 3)]
    return [v[i:i + 4] for i in range(0, len(v), 4)]


def test_which_layers_run_in_one_launch(tmp_path):
    """the shapes of tests/test_gpu_direct.py run where that file has them run"""
    from tests.test_gpu_direct import BEYOND, FC, FC_LINES, LAYERS, LINES, SPLITS
    two = {(2, 129, 3, 40, 40, 3, 3, 0, 3), (1, 64, 17, 17, 31, 7, 7, 3, 1)} | set(LINES[4:6] + LINES[7:10] + LINES[11:12] + LINES[13:]) | set(BEYOND)
    layers = LAYERS + LINES + list(SPLITS) + BEYOND
    for layer, plan in zip(layers, _plans(tmp_path, layers)):
        assert [p[0] for p in plan] == [layer not in two] * 4, layer
        if layer in SPLITS:
            assert plan[0][1:] == SPLITS[layer], (layer, plan)
    # fully connected: pieces of input, then records of binary weights beyond 8 MiB
    fc = FC + FC_LINES
    plans = _plans(tmp_path, [(n, c, 1, 1, kn, 1, 1, 0, 1) for n, c, kn in fc])
    for layer, plan in zip(fc, plans):
        runs = [True] * 4 if layer not in FC_LINES[1:3] else [False] * 4
        if layer == FC_LINES[-1]:
            runs = [True, False, True, False]
        assert [p[0] for p in plan] == runs, layer


def test_layers_that_measured_slower_in_one_launch(tmp_path):
    slow = [(36, 44, 2, 2, 942, 5, 5, 2, 1), (38, 245, 6, 6, 636, 3, 3, 0, 2), (23, 178, 5, 5, 1432, 5, 5, 0, 1), (29, 44, 3, 3, 1295, 7, 7, 3, 2), (14, 110, 5, 5, 1169, 3, 3, 1, 1),
            (22, 160, 2, 2, 1109, 5, 5, 2, 1), (29, 36, 3, 3, 1638, 3, 3, 0, 2), (3, 79, 28, 28, 227, 5, 2, 2, 1), (2, 69, 23, 23, 388, 5, 2, 2, 1)]
    faster = [(8, 128, 28, 28, 128, 3, 3, 1, 1), (24, 64, 14, 14, 256, 3, 3, 1, 1), (1, 64, 16, 16, 256, 3, 3, 1, 1), (3, 64, 39, 39, 256, 1, 1, 0, 1)]
    assert [p[0][0] for p in _plans(tmp_path, slow)] == [False] * len(slow)
    assert [p[0][0] for p in _plans(tmp_path, faster)] == [True] * len(faster)


def test_cut_of_layers(tmp_path):
    """the shapes of tests/test_gpu_deep_layers.py stand on the sides of the lines that they are there for: eight wavefronts on one tile from
    75 words on and up to 256 tiles of 32 x 32, never with a split forced or a hand-over"""
    from tests.test_gpu_deep_layers import LAYERS
    deep = [layer not in (LAYERS[0], LAYERS[7], LAYERS[-1]) for layer in LAYERS]
    assert not any(p[0] for plan in _plans(tmp_path, LAYERS) for p in plan)   # none in one launch
    rows = []
    for n, c, h, w, kn, kh, kw, pad, stride in LAYERS:
        oh, ow = (h + 2 * pad - kh) // stride + 1, (w + 2 * pad - kw) // stride + 1
        rows.append((n * oh * ow, kn, -(-c // 64) * kh * kw))
    out = _run(tmp_path, r"""
int main() {
    const long v[][3] = {""" + ", ".join("{%d, %d, %d}" % r for r in rows) + r"""};
    for (auto& l : v) {
        const LayerCut c = layer_cut(l[0], l[1], l[2], false, 0, -1);
        if (layer_cut(l[0], l[1], l[2], true, 0, -1).deep || layer_cut(l[0], l[1], l[2], false, 4, -1).deep || (c.deep && !c.small)) return 1;
        printf("%d ", c.deep);
    }
    // every split keeps a pair of words for each wavefront; results with few tiles take small ones
    for (long tiles : {1, 149, 150, 299, 300, 449, 450, 519, 520, 599, 600, 799, 800, 1023, 1024, 1499, 1500})
        for (int K : {1, 2, 3, 4, 5, 8, 39, 40, 119, 120})
            for (bool hand_over : {false, true}) {
                const LayerCut c = layer_cut(64 * tiles, 64, K, hand_over, 0, -1);
                const long from1 = hand_over ? 600 : K >= 40 ? 1500 : 1024, from2 = hand_over ? 450 : K >= 40 ? 800 : 520;
                const int want = tiles >= from1 ? 1 : tiles >= from2 ? 2 : 4;
                if ((K + 1) / 2 < c.split || c.split > want || ((K + 1) / 2 >= want && c.split != want)) return 2;
                if (c.small != (tiles < (hand_over || K >= 120 ? 150 : 300))) return 3;
            }
}
""")
    assert [v == "1" for v in out.split()] == deep, list(zip(LAYERS, rows, out.split()))
