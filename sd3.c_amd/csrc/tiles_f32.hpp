// Which tile shape a launch of fp32 products takes. Host code only.
#pragma once

namespace sd3 {

// The tile shapes, largest first, and what one K tile (32 k values) of one output tile costs in cycles, measured over N = 1536 .. 6144
// and K = 1536, 6144: alone on its compute unit, and with two or three workgroups sharing one (the matrix instructions alone: TM*TN/4).
struct F32Tile {
    int tm, tn;
    double alone, shared;
};
constexpr int F32_TILES = 5;
constexpr F32Tile f32_tiles[F32_TILES] = {{128, 128, 4270, 4250}, {128, 64, 2150, 2155}, {64, 64, 1150, 1100}, {32, 64, 670, 590}, {32, 32, 440, 325}};
// The same for depths that are not whole K tiles, whose loads have 64-bit addresses (K = 1548, 6156): the small tiles issue more of them per matrix
// instruction and lose more. Chosen by the table above 1178 x 6144 x 1548 took 32x64 tiles, 207 us (128x128: 194), 6000 x 4608 x 1548 64x64 ones, 694
// (660), 1178 x 6144 x 780 122 (109).
constexpr F32Tile f32_tiles_ragged_k[F32_TILES] = {{128, 128, 4690, 4660}, {128, 64, 2560, 2430}, {64, 64, 1420, 1300}, {32, 64, 890, 720}, {32, 32, 580, 410}};

struct F32Layer {
    int M, N, K;
};
// The shape whose busiest compute unit is done first: with r output tiles on it, r * shared cycles per K tile (alone for r = 1).
inline int pick_f32_tile(const F32Layer* layers, int n, int cus, bool whole_k) {
    int best = 0;
    double best_cost = 0;
    for (int s = 0; s < F32_TILES; s++) {
        const F32Tile t = whole_k ? f32_tiles[s] : f32_tiles_ragged_k[s];
        long long tiles = 0, depth = 0;
        for (int i = 0; i < n; i++) {
            const long long c = (long long)((layers[i].M + t.tm - 1) / t.tm) * ((layers[i].N + t.tn - 1) / t.tn);
            tiles += c;
            depth += c * layers[i].K;
        }
        const long long r = (tiles + cus - 1) / cus;
        const double cost = (double)depth / tiles * (r == 1 ? t.alone : r * t.shared);
        if (s == 0 || cost < best_cost) {
            best = s;
            best_cost = cost;
        }
    }
    return best;
}

}  // namespace sd3
