// Which tiles a prefill product runs on: host arithmetic only.
#pragma once

namespace yuf {

// Forms of gemm_ps_kernel: fp32 products from W planes, fp32 products that split
// W as they go, bf16 W, and fp32 MFMA.
enum PsMode : int { PS_X3P = 0, PS_X3 = 1, PS_BF16 = 2, PS_F32 = 3 };

// A tile shape and the measured time (us) of one 32-k step of it: of tiles that
// have their CUs to themselves, and of each full round of 256 tiles.
struct TileCost {
    int id, bm, bn;
    float alone, round;
};
// gemm_ps_kernel's tiles per mode.
constexpr TileCost kPsTiles[4][4] = {
    {{1, 32, 32, 0.30f, 0.168f}, {2, 64, 64, 0.60f, 0.45f}, {3, 128, 128, 1.22f, 1.31f}, {}},                        // PS_X3P
    {{1, 32, 32, 0.35f, 0.20f}, {2, 64, 64, 0.70f, 0.48f}, {3, 128, 128, 1.65f, 1.65f}, {}},                         // PS_X3
    {{1, 32, 32, 0.23f, 0.10f}, {2, 64, 64, 0.32f, 0.205f}, {3, 128, 128, 0.64f, 0.65f}, {4, 64, 128, 0.47f, 0.34f}},  // PS_BF16
    {{1, 32, 32, 0.24f, 0.195f}, {2, 64, 64, 0.67f, 0.55f}, {5, 32, 64, 0.40f, 0.33f}, {}},                          // PS_F32
};
// The 256-row tiles of the same forms (64-wide X3P: 64-row tiles), widths 256, 160, 128, 64.
constexpr TileCost kBigTiles[3][4] = {
    {{0, 256, 256, 3.55f, 4.3f}, {0, 256, 160, 2.4f, 3.0f}, {0, 256, 128, 2.05f, 2.4f}, {0, 64, 64, 0.47f, 0.40f}},
    {{0, 256, 256, 4.0f, 4.4f}, {0, 256, 160, 2.8f, 3.0f}, {0, 256, 128, 2.3f, 2.6f}, {0, 256, 64, 1.9f, 2.2f}},
    {{0, 256, 256, 1.6f, 1.95f}, {0, 256, 160, 1.2f, 1.7f}, {0, 256, 128, 1.05f, 1.6f}, {0, 256, 64, 0.87f, 1.5f}},
};

struct TileProduct {
    int rows, N;  // rows over all parts of a call that run side by side
};

// The tile of gemm_ps_kernel that a group of n products (deepest K) takes, or
// nullptr: the 256-row tiles of width big_bn (0: there are none).  The estimate
// of a launch is its rounds of 256 tiles times the measured time of a k step;
// tiles are counted over the rows of the whole call, since a prefill's parts run
// side by side.  us under a sustained load, this kernel's best tile against the 256-row
// tiles: X3P 333 x 640 x 640 9 / 50, 333 x 640 x 2560 26 / 183, 1000 x 5120 x
// 640 45 / 76, 4000 x 5120 x 640 133 / 163, 5000 x 5120 x 640 173 / 169, 16384 x
// 5120 x 640 503 / 468; X3 1300 x 8192 x 1024 158 / 138, 12000 x 1024 x 4096 625 /
// 514; bf16 2200 x 1024 x 4096 65 / 199, 16384 x 1024 x 4096 330 / 259.  Over 400
// shapes of 300 to 16384 rows the rule is 1 % off the best tile on average.
// X3P products with K <= 128 move to it below 2048 rows only: there the output
// write bounds both (640 x 128: 6.3 / 8.1 at 1000 rows, 11 / 9.8 at 4096).  Where
// the X3P kernel's widest tile is 64 x 64, that form beats this one's of the same
// size (three products 16384 x 64 x 640 44 / 53, 16384 x 448 x 640 62 / 69).
inline const TileCost *ps_tile_rule(const TileProduct *p, int n, int K, int mode, int big_bn, bool silu) {
    int rows = 0;
    bool n128 = true;
    for (int i = 0; i < n; ++i) {
        rows = p[i].rows > rows ? p[i].rows : rows;
        n128 = n128 && p[i].N % 128 == 0;
    }
    if (mode == PS_X3P && K <= 128 && rows >= 2048 && big_bn) return nullptr;
    const auto cost = [&](const TileCost &t) {
        long long tiles = 0;
        for (int i = 0; i < n; ++i) tiles += (long long)((p[i].rows + t.bm - 1) / t.bm) * ((p[i].N + t.bn - 1) / t.bn);
        if (tiles <= 256) return t.alone >= t.round ? t.alone : t.alone + (t.round - t.alone) * (float)tiles / 256.0f;
        const float rounds = t.round * (float)((tiles + 255) / 256);
        return t.alone > rounds ? t.alone : rounds;
    };
    const TileCost *best = nullptr;
    float least = 0.0f;
    if (big_bn && mode != PS_F32)
        for (const TileCost &t : kBigTiles[mode])
            if (t.bn == big_bn) least = cost(t);
    for (const TileCost &t : kPsTiles[mode]) {
        if (!t.id || (silu && t.bn < 64) || (t.bn == 128 && !n128)) continue;
        if (mode == PS_X3P && big_bn == 64 && t.bn == 64) continue;
        const float c = cost(t);
        if (least == 0.0f || c < least) {
            least = c;
            best = &t;
        }
    }
    return best;
}

}  // namespace yuf
