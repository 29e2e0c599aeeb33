"""Where the layer kernel looks for the record of every K word (fastertnn_amd/csrc/pair_walk.h, the code the kernel runs), against the
word's place in 64-bit arithmetic: even and odd numbers of channel words, windows of one and several taps, every K split, both
lane halves, images from a few pixels up to the 2^31 records a call's operand may have.  CPU only."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

_PROGRAM = r"""
#include <stdio.h>
#include <stdlib.h>
#include <initializer_list>
#include "pair_walk.h"
using namespace ftnn;
static long checked = 0, beyond = 0;   // records compared; of these, scalar parts of 4 GiB and more

template <uint32_t UNIT, bool FIRST>
void share(const PairWalk& pw, const ConvGeom& cg, int64_t img, int ih0, int iw0, int p0, int p1, int h) {
    const int64_t HW = (int64_t)cg.H * cg.W;
    const uint32_t xrec = (uint32_t)img * (uint32_t)(cg.CP * cg.H * cg.W) + (uint32_t)(ih0 * cg.W + iw0);
    PairPos<UNIT> pos;
    pos.template start<FIRST>(pw, cg, p0, h);
    uint32_t rec = xrec + pos.off(cg);
    for (int p = p0; p < p1; p++) {
        const int w = 2 * p + h, tap = w / cg.CP, ic = w % cg.CP, kh = tap / cg.KW, kw = tap % cg.KW;
        const bool real = w < cg.K;
        if (real != (pos.kh < pw.KH) || pos.kh != kh || pos.kw != kw) { printf("tap of word %d, %d words of channels\n", w, cg.CP); exit(1); }
        const int ih = ih0 + kh, iw = iw0 + kw;
        if (real && ih >= 0 && ih < cg.H && iw >= 0 && iw < cg.W) {
            const int64_t want = (img * cg.CP + ic) * HW + (int64_t)ih * cg.W + iw;
            const int64_t got = (int64_t)((uint64_t)rec + pos.soff / UNIT);
            if (pos.soff % UNIT != 0 || got != want) {
                printf("word %d of %d x %d x %d words: record %lld, not %lld\n", w, cg.CP, cg.H, cg.W, (long long)got, (long long)want);
                exit(1);
            }
            checked++;
            beyond += (int64_t)(pos.soff / UNIT) * 16 >= (1LL << 32);
        }
        if (p + 1 < p1 && pos.next(pw, cg)) rec = xrec + pos.off(cg);
    }
}

template <uint32_t UNIT>
void layer(int CP, int H, int W, int KH, int KW, int pad, int64_t images) {
    ConvGeom cg = {H, W, CP, 0, 0, KW, CP * KH * KW, pad, pad, 1, 1, make_fastdiv(1), make_fastdiv((uint32_t)CP), make_fastdiv((uint32_t)KW)};
    const PairWalk pw = make_pair_walk(cg);
    const int places[3][2] = {{-pad, -pad}, {H - KH + pad, W - KW + pad}, {H / 2, W / 3}};
    for (auto& at : places)
        for (int64_t img : {(int64_t)0, images - 1})
            for (int h = 0; h < 2; h++) {
                share<UNIT, true>(pw, cg, img, at[0], at[1], 0, pw.NP, h);
                for (int S : {2, 4, 8})
                    for (int ks = 0; ks < S; ks++)
                        share<UNIT, false>(pw, cg, img, at[0], at[1], (int)((uint32_t)(pw.NP * ks) / S), (int)((uint32_t)(pw.NP * (ks + 1)) / S), h);
            }
}

int main() {
    const int sides[][2] = {{7, 5}, {56, 56}, {1024, 1000}, {8192, 4096}, {8190, 8190}, {1, 67000000}, {67000000, 1}};
    const int windows[][3] = {{1, 1, 0}, {3, 3, 1}, {1, 2, 0}, {3, 1, 2}, {5, 7, 0}};
    for (auto& s : sides)
        for (auto& k : windows)
            for (int CP : {1, 2, 3, 4, 5, 6, 7, 8, 10, 11, 16, 25, 31, 32}) {
                const int64_t recs = (int64_t)CP * s[0] * s[1], images = 0x7fffffffLL / recs;
                if (images < 1 || (int64_t)(s[0] + 2 * k[2]) * (s[1] + 2 * k[2]) >= (1 << 26) || s[0] + 2 * k[2] < k[0] || s[1] + 2 * k[2] < k[1]) continue;
                layer<1>(CP, s[0], s[1], k[0], k[1], k[2], images < 65535 ? images : 65535);
                const int64_t in_buffer = 0xf0000000LL / 16 / recs;   // images of an operand that buffer loads take
                if (in_buffer >= 1) layer<16>(CP, s[0], s[1], k[0], k[1], k[2], in_buffer < 65535 ? in_buffer : 65535);
            }
    printf("ok %ld %ld\n", checked, beyond);
    return 0;
}
"""


def test_every_word_of_every_share_is_found(tmp_path):
    src, exe = tmp_path / "walk.cpp", tmp_path / "walk"
    src.write_text(_PROGRAM)
    subprocess.run(["g++", "-O1", "-std=c++17", "-fsanitize=undefined", "-fno-sanitize-recover=all", "-I", os.path.join(ROOT, "fastertnn_amd", "csrc"),
                    str(src), "-o", str(exe)], check=True, timeout=120)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-500:] + r.stderr[-500:]
    ok, checked, beyond = r.stdout.split()
    assert ok == "ok" and int(checked) > 50000 and int(beyond) > 1000   # (the sizes above reach past 4 GiB within an image)
