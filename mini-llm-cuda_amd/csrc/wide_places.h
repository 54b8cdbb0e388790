// Which pieces of its operands a wave of k_decode_wide loads, and the flags it waits for first (kernels_wide.hip).  A piece that is loaded and multiplied, also by
// weights of zero (0 x NaN is NaN), has to be among those waited for: tests/test_wide_places.py goes through all shapes on the CPU.
#pragma once

#define WD_WAVES 8
#define WD_CA 3 // chunks of 32 columns a wave has of a product over the whole width: dim <= 768

constexpr int wd_min(int a, int b) { return a < b ? a : b; }

// A product over the whole width of nch chunks: chunks wave, wave + 8, ... are a wave's, `cnt` of them; past its last one the last once more.
constexpr int wd_count(int wave, int nch) { return (nch - wave + WD_WAVES - 1) / WD_WAVES; }
constexpr int wd_chunk(int wave, int k, int cnt) { return wave + WD_WAVES * wd_min(k, cnt - 1); }
// The flag of lane `lane` (a flag per tile of 16 columns and block of 16 tokens, mb blocks in all): its chunks' tiles, mw blocks from block0 on.
constexpr int wd_flag1(int lane, int wave, int cnt, int mb, int mw, int block0) {
    const int i = wd_min(lane, cnt * 2 * mw - 1), c = i / (2 * mw), j = i - c * 2 * mw;
    return (wd_chunk(wave, c, cnt) * 2 + j / mw) * mb + block0 + j % mw;
}
// Output and down projection: chunks part, part + 4 of `count`, past the last one that.
constexpr int wd_part(int part, int i, int count) { return wd_min(part + 4 * i, count - 1); }
// Mixing output: a chunk is half a head (4 units of 16 rows a head, a flag per unit and sequence), behind the heads the PLE columns (a flag per block).
// The first unit of chunk wd_part(part, i, count); a second head without sequences stands for the first one.
constexpr int wd_mix_chunk(int part, int i, int count, int nh, bool none) {
    const int c = wd_part(part, i, count);
    return none && c >= 2 && c < nh * 2 ? c - 2 : c;
}
constexpr int wd_flagM(int lane, int c, int from, int to) { return ((c >> 1) * 4 + (c & 1) * 2) * 64 + wd_min(from + lane, to - 1); }
// FFN units: a flag per tile of 8 units and block of tokens.
constexpr int wd_flagU(int lane, int part, int count, int mb) {
    const int i = wd_min(lane, 8 * mb - 1);
    return wd_part(part, i / (4 * mb), count) * 4 * mb + i % (4 * mb);
}
