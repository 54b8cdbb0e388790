// Every piece of an operand that a wave of k_decode_wide loads and multiplies lies behind flags it has waited for, over all shapes the kernel covers.
#include <cstdio>
#include <set>

#include "wide_places.h"

static int bad = 0;
static void need(bool ok, const char* what, int a, int b, int c, int d) {
    if (!ok && bad++ < 10) printf("%s: %d %d %d %d\n", what, a, b, c, d);
}

int main() {
    long seen = 0;
    for (int nch : {16, 20, 24})              // dim 512, 640, 768
        for (int mb = 1; mb <= 4; mb++) {     // blocks of 16 tokens
            const int ts = mb == 4 ? 2 : 1, mw = mb / ts;
            for (int wave = 0; wave < WD_WAVES; wave++)
                for (int half = 0; half < ts; half++) { // residual planes and their sums of squares
                    const int cnt = wd_count(wave, nch), block0 = half * mw;
                    std::set<int> waited, mine;
                    for (int lane = 0; lane < 64; lane++) waited.insert(wd_flag1(lane, wave, cnt, mb, mw, block0));
                    for (int k = 0; k < WD_CA; k++) {
                        const int chunk = wd_chunk(wave, k, cnt);
                        need(chunk < nch, "chunk", nch, wave, k, chunk);
                        if (k < cnt) mine.insert(chunk);
                        for (int tile = 2 * chunk; tile < 2 * chunk + 2; tile++)
                            for (int b = block0; b < block0 + mw; b++, seen++) need(waited.count(tile * mb + b), "width", nch, mb, wave, k);
                    }
                    need((int)mine.size() == cnt && (wave >= nch || cnt >= 1) && cnt <= WD_CA, "count", nch, mb, wave, cnt);
                }
            for (int count = 1; count <= 8; count++) // FFN units
                for (int part = 0; part < 4; part++) {
                    std::set<int> waited;
                    for (int lane = 0; lane < 64; lane++) waited.insert(wd_flagU(lane, part, count, mb));
                    for (int i = 0; i < 2; i++)
                        for (int tile = 0; tile < 4; tile++)
                            for (int b = 0; b < mb; b++, seen++) need(waited.count((wd_part(part, i, count) * 4 + tile) * mb + b), "units", mb, count, part, i);
                }
        }
    for (int heads : {8, 10, 12}) // mixing output: tokens of a second head that another XCD has are not multiplied
        for (int n = 1; n <= 64; n++)
            for (int X = 0; X < 8; X++)
                for (int ple = 0; ple < 2; ple++) {
                    const int second = heads - 8, nh = second > 0 ? 2 : 1, count = nh * 2 + ple;
                    int lo = 0, hi = 0;
                    if (second > 0) {
                        const int sharers = (8 - X % second + second - 1) / second;
                        lo = n * (X / second) / sharers;
                        hi = n * (X / second + 1) / sharers;
                    }
                    for (int part = 0; part < 4; part++) {
                        std::set<int> waited;
                        bool blocks = false; // ... the PLE columns' flags
                        for (int i = 0; i < 2; i++) {
                            const int c = wd_mix_chunk(part, i, count, nh, lo >= hi);
                            if (c >= nh * 2) blocks = true;
                            else
                                for (int lane = 0; lane < 64; lane++)
                                    for (int unit = 0; unit < 2; unit++) waited.insert(wd_flagM(lane, c, c >> 1 ? lo : 0, c >> 1 ? hi : n) + unit * 64);
                        }
                        for (int i = 0; i < 2; i++) {
                            const int c = wd_part(part, i, count), hl = c >> 1;
                            if (c >= nh * 2) { need(blocks, "columns", heads, n, X, part); continue; }
                            for (int tok = hl ? lo : 0; tok < (hl ? hi : n); tok++, seen++)
                                for (int unit = (c & 1) * 2; unit < (c & 1) * 2 + 2; unit++) need(waited.count((hl * 4 + unit) * 64 + tok), "mixing", heads, n, X, part);
                        }
                    }
                }
    printf("%ld pieces, %d not waited for\n", seen, bad);
    return bad != 0;
}
