// How the chunked WKV-7 scan spreads heads over workgroups: host arithmetic only.
#pragma once

namespace yuf {

constexpr int kWkvCus = 256;  // workgroups of the scan that run at once: one fits a CU

// Value tiles of a workgroup for heads of NB tiles of 16 value rows: 0 whole
// heads, 1 a workgroup per tile, (NB + 1) / 2 two workgroups per head (`two`:
// that form exists).  A finer split repeats the key-space stages but shortens the
// busiest SIMD of a chunk, so it pays while every workgroup runs at once, counted
// over the heads of the whole call (`all`), since a prefill's parts run side by
// side.  us for 777 tokens, whole / two / one per tile: N = 64, 48 heads 130 / 104 /
// 85, 80 heads 129 / 107 / 163, 128 heads 132 / 111 / 171, 192 heads 137 / 211 /
// 245; N = 40, 16 heads 78 / 64.9 / 63.3, 80 heads 80.6 / 68.2 / 67.1, 128 heads
// 83 / 71 / 126.  us of a prefill in parts (N = 40, 4 layers, 2048 tokens): 128
// heads in four 6260 / 6150 / 6180, 160 in two 5610 / 5720 / 6070, 256 in two
// 8190 / 8580 / 8950.  N = 64 with the model's prep has no pair form; its parts'
// scans seldom coincide, so one per tile pays up to two rounds of the CUs in all
// (2 layers, 1111 tokens, whole / one per tile: 96 heads in four 2200 / 2040, 128
// in four 2440 / 2375, 192 in two 2370 / 2550).
inline int wkv7_value_tiles(int NB, int heads, int all, bool two, const char *force) {
    // Of the forcing texts "0", "2" and "4" name a form; any other one means split.
    int forced = -1;
    if (force) forced = (force[0] == '0' || force[0] == '2' || force[0] == '4') && !force[1] ? force[0] - '0' : 1;
    if (NB < 2 || forced == 0) return 0;
    const int pair = (NB + 1) / 2;
    if (forced == 4) return 1;
    if (forced == 2) return two ? pair : 0;
    if (all < heads) all = heads;
    if (all * NB <= kWkvCus) return 1;
    if (two) return forced > 0 || all * 2 <= kWkvCus ? pair : 0;
    return heads * NB <= kWkvCus && all * NB <= 2 * kWkvCus ? 1 : 0;
}

}  // namespace yuf
