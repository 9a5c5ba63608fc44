// Which kernel and tile shape a launch of fp32 products takes. Host code only.
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

// ---- products of bf16 pieces (gemm_f32_pieces_kernel) ----
// Which launches: depths of 512 and more, in whole groups of the four K tiles that its loops take at a time. us, fp32 instruction | pieces: over 1 to 8192 rows, 256 to 6144
// columns the mean is 0.93 of the fp32 instruction's time at K = 512, 0.90 from 768 on, 0.96 at 256, where large products gain (8192 x 1536 57 | 49) and small ones lose, which
// are what such models consist of (width 256, 2 heads, three blocks, 1178 tokens: a forward 327 us, with pieces from K = 256 on 334). One round of small
// tiles is up to a tenth slower (154 x 1536 x 1536 12.9 | 13.8, 666 x 1536 x 1536 29.4 | 30.5), from 1178 rows and 768 columns on it is 0.6 to 0.9. By the depth alone: the two kernels
// round differently, and a row's result is to be the same in every batch.
inline bool f32_by_pieces(const F32Layer* layers, int n) {
    for (int i = 0; i < n; i++)
        if (layers[i].K % 128 || layers[i].K < 512) return false;
    return true;
}

// The shapes (the first five as above) and their times in us, measured over M = 1 .. 8192, N = 768 .. 6144 and K = 256 .. 6144 (to 2 to 9 %): a launch's last round apart from its K tiles, each
// round before it likewise, a K tile of a lone workgroup, and by how much longer that takes with every compute unit at work (the power limit; it grows with
// the square of the share that is).
struct F32PieceTile {
    int tm, tn;
    double last, before, step, crowd;
};
constexpr int F32_PIECE_TILES = 6;
constexpr F32PieceTile f32_piece_tiles[F32_PIECE_TILES] = {{128, 128, 6.7, 5.2, 0.954, 0.32}, {128, 64, 6.1, 3.8, 0.538, 0.32}, {64, 64, 6.3, 2.9, 0.309, 0.32},
                                                           {32, 64, 6.5, 0.7, 0.227, 0.11},    {32, 32, 6.5, 0.5, 0.154, 0.04},  {256, 128, 8.6, 5.7, 1.860, 0.35}};
// The same where A comes in pieces. (1178 and 333 rows of 1536 columns, K = 1536 and 6144, 1178 to 18848 of 2304 to 6144, K = 768 and 1536. 40 blocks of
// other widths from 512 to 3072, expansions and rows: 0.90 to 1.01 of their time with the fastest one shape in all of their products)
constexpr F32PieceTile f32_a_piece_tiles[F32_PIECE_TILES] = {{128, 128, 9.2, 6.5, 0.890, 0.22}, {128, 64, 7.9, 3.7, 0.562, 0.22}, {64, 64, 6.4, 0.8, 0.404, 0.04},
                                                             {32, 64, 6.4, 0.7, 0.235, 0.10},  {32, 32, 7.0, 0.3, 0.150, 0.06},  {256, 128, 14.0, 10.5, 1.390, 0.36}};
inline int pick_f32_piece_tile(const F32Layer* layers, int n, int cus, const F32PieceTile* shapes = f32_piece_tiles) {
    int best = 0;
    double best_cost = 0;
    for (int s = 0; s < F32_PIECE_TILES; s++) {
        const F32PieceTile t = shapes[s];
        long long tiles = 0, depth = 0;
        for (int i = 0; i < n; i++) {
            const long long c = (long long)((layers[i].M + t.tm - 1) / t.tm) * ((layers[i].N + t.tn - 1) / t.tn);
            tiles += c;
            depth += c * layers[i].K;
        }
        const long long full = (tiles - 1) / cus;
        const double part = (double)(tiles - full * cus) / cus, steps = (double)depth / tiles / 32 * t.step;
        const double cost = full * (t.before + steps * (1 + t.crowd)) + t.last + steps * (1 + t.crowd * part * part);
        if (s == 0 || cost < best_cost) {
            best = s;
            best_cost = cost;
        }
    }
    return best;
}

}  // namespace sd3
