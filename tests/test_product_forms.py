"""Which form of a matrix-core product runs (fastertnn_amd/csrc/product_forms.h, the code the launchers run): the forms that the
shapes of the GPU tests are there for, and the choice between estimates that say the same.  CPU only."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def choose(tmp_path_factory):
    """(images, OH, OW, columns, words) of each product -> (whether whole calls of 160 tiles and more run from the rows, form of k_rows, form of kept operands)"""
    tmp = tmp_path_factory.mktemp("forms")
    src, exe = tmp / "forms.cpp", tmp / "forms"
    src.write_text(r"""
#include <stdio.h>
#include "product_forms.h"
using namespace ftnn;
int main() {
    long long n, oh, ow;
    int kn, kw;
    while (scanf("%lld %lld %lld %d %d", &n, &oh, &ow, &kn, &kw) == 5) {
        const long long M = n * oh * ow, OHW = oh * ow, p = OHW > 1 ? kn : M, q = OHW > 1 ? M : kn;
        if (M > 0x7fffffffLL) printf("%d 0 0\n", mm_rows_within_limits(M, kn, kw));   // (no such product is launched)
        else printf("%d %d %d\n", mm_rows_ahead_of_packing(M, OHW, kn, kw), rows_form(p, q, kw), packed_form(p, q, kw / 2));
    }
}
""")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fsanitize=undefined", "-fno-sanitize-recover=all", "-I", os.path.join(ROOT, "fastertnn_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True, timeout=120)

    def run(shapes):
        r = subprocess.run([str(exe)], input="\n".join("%d %d %d %d %d" % s for s in shapes), capture_output=True, text=True, check=True, timeout=120)
        return [tuple(int(v) for v in line.split()) for line in r.stdout.splitlines()]

    return run


def test_a_tie_keeps_the_smaller_tile(choose):
    """products that measured 15 to 20 % slower by the least estimate, and products whose estimates are further apart or of other forms"""
    ties = {(752, 1, 1, 459, 1532): 0, (563, 1, 1, 483, 1456): 0, (334, 1, 1, 811, 1528): 0, (186, 1, 1, 2684, 1768): 0, (61, 1, 1, 6236, 1644): 0, (85, 1, 1, 3094, 1608): 0}
    clear = {(896, 1, 1, 873, 20): 4, (240, 1, 1, 5957, 24): 4, (332, 1, 1, 8180, 4): 4, (2506, 1, 1, 1365, 8): 4, (3328, 1, 1, 3328, 16): 6, (1024, 1, 1, 1024, 128): 1, (1999, 1, 1, 1733, 228): 3, (1, 1, 1, 7660, 120): 5}
    for shapes in (ties, clear):
        assert {s: c[1] for s, c in zip(shapes, choose(shapes))} == shapes


def test_shapes_of_the_gpu_test_run_the_forms_they_are_there_for(choose):
    from tests.test_gpu_product_forms import FORMS
    reached = {"rows": {}, "kept": {}}
    for (n, oh, ow, kn, kw), want, got in zip(FORMS, FORMS.values(), choose(list(FORMS))):
        m, row = n * oh * ow, oh * ow if oh * ow > 1 else kn
        small = -(-m // 256) * -(-kn // 256) < 160 or kn < 128 or m < 128   # from packed rows without an estimate (mm_from_rows)
        assert (got[1] if small or got[0] else 7, got[2]) == want, (n, oh, ow, kn, kw)
        past = row % 16 == 0 or m * kn <= 4 << 20   # stores_past_caches
        for side, form in zip(("rows", "kept"), want):
            reached[side].setdefault(form, set()).update((past, "nchw" if oh * ow > 1 else "row-major"))
    # forms on up to 256 tiles of 32 x 32 have no large results, nor does any choice of 32 x 32 on four wavefronts
    small_only = {"rows": (0, 5), "kept": (0, 1)}
    for side, count in (("rows", 8), ("kept", 10)):
        for form in range(count):
            want = {True, "nchw", "row-major"} | (set() if form in small_only[side] else {False})
            assert reached[side][form] == want, (side, form)


def test_limits_of_sizes_that_no_call_launches(choose):
    """rows up to the largest that a size query may name: refused without an overflow (the program above is built to end there)"""
    last = 0x7fffffff
    assert choose([(last, last, 1, last, 4), (last, last, 1, 1, 4), (1 << 31, 1, 1, 1, 4), (last, 1, 1, 1, 4)])[:3] == [(0, 0, 0)] * 3
    assert choose([(last, 1, 1, last, 4)])[0][0] == 0 and choose([(16777208 * 128, 1, 1, 1, 4)])[0][0] == 1
