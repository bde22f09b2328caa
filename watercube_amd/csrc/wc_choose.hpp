// wc_choose.hpp -- choices by size, density and times, as plain functions of numbers: the box shape of the tile passes,
// whether a context starts with them, which boxes are thin, and the tuner's candidates.  Host code without HIP.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <math.h>

#include <vector>

namespace wc {

// Tile passes (the last variant): a workgroup stages one box of cells and its halo in LDS.
struct TileShape {
    int x, y, z;  // cells of a base box
    int block;    // threads per workgroup: kTileLargeBlock or kTileSmallBlock
    int cap;      // records (box and halo) its LDS holds
};
constexpr int kTileLargeBlock = 512, kTileLargeCap = 1920;
constexpr int kTileSmallBlock = 256, kTileSmallCap = 2304;

// Neighbours a particle's list holds (16 bits each; particles with more search directly): dense clusters
// have a few hundred; large contexts keep lists of half the size.
inline uint32_t tile_list_cap(uint64_t particles) {
    return particles <= 500000 ? 512u : particles <= 4000000 ? 256u : 128u;
}

// What a scene's parameters say of its density.
struct SceneFill {
    double n;           // particles
    double rest;        // particles a cell holds at rest density (0: the parameters name none)
    double occupancy;   // the same, or the grid's mean where that is more
    double neighbours;  // within the kernel radius, at the larger of the two densities
};
inline SceneFill scene_fill(uint32_t n, int grid_res, double bin, double h, double rest_density, double mass) {
    const double cell = bin * bin * bin, mean = (double)n / ((double)grid_res * grid_res * grid_res);
    SceneFill f{(double)n, 0.0, 0.0, 0.0};
    const double rest = rest_density / mass * cell;
    if (rest > 0.0 && rest < 1e6) f.rest = rest;
    f.occupancy = f.rest > mean ? f.rest : mean;
    const double ball = 4.18879 * (h / bin) * (h / bin) * (h / bin);
    f.neighbours = f.occupancy * (ball < 27.0 ? ball : 27.0);
    return f;
}

// Base box of the tile passes.  Larger boxes stage less halo per particle; they have to fit LDS at rest density (a
// denser one is split) and leave the chip's 256 CUs enough boxes each.  At 8 particles a cell the whole step took, by
// 4x3x4 / 4x2x4 / 2x2x4 (us): 91,125 particles 141 / 130 / 104, 125,000 126 / 137 / 137, 262,144 141 / 158 / 176: the
// first from 300 boxes of it.  At 12 a cell, where it does not fit, by 4x2x4 / 2x2x4: 125,000 182 / 135, 192,089 (once
// spread, three at once) 94 / 111, 2,048,000 1,087 / 1,109: the second from 450 boxes.  Up to 16 a cell 2x2x4
// otherwise.  Above, where a box of it has more particles than threads, by 2x2x4 / 2x2x2: 59,319 (20 a cell) 192 / 143,
// 125,000 (20) 249 / 234, 343,000 (19) 553 / 542, 704,969 (17) 969 / 1,071, 1,000,000 (19) 1,321 / 1,388, 4,492,125
// (19) 5,762 / 6,093: 2x2x2 below 2,000 boxes of 2x2x4.
inline TileShape choose_tile_shape(const std::vector<SceneFill>& scenes) {
    double n = 0.0, cell = 0.0;
    for (const SceneFill& f : scenes) {
        n += f.n;
        cell += f.rest * f.n;
    }
    cell = n > 0.0 ? cell / n : 0.0;
    const struct {
        TileShape t;
        double boxes;
    } shapes[] = {{{4, 3, 4, kTileLargeBlock, kTileLargeCap}, 300.0},
                  {{4, 2, 4, kTileLargeBlock, kTileLargeCap}, 450.0},
                  {{2, 2, 4, kTileSmallBlock, kTileSmallCap}, 2000.0}};
    for (const auto& s : shapes) {
        const TileShape& t = s.t;
        if ((t.x + 2) * (t.y + 2) * (t.z + 2) * cell * 1.05 <= t.cap && n >= s.boxes * (t.x * t.y * t.z) * cell)
            return t;
    }
    return {2, 2, 16.0 * cell <= kTileSmallBlock ? 4 : 2, kTileSmallBlock, kTileSmallCap};
}

// Contexts of this many particles start with the tile passes.  Smaller ones gain while the fluid is at rest
// density (16,384 particles, three contexts at once: 20 us a step against 33) and lose as it spreads and boxes
// empty (44 against 36 at step 4,000); 80,000 particles gain in both (83 against 131, 84 against 122).
// Batches also need 20,000 particles a scene: 62 scenes of about 31,000 780 -> 693, 28 of about 14,000 207 -> 215
// once spread.  wc_tune times both whatever the size.
constexpr uint32_t kTileMinParticles = 50000, kTileMinPerScene = 20000;

// Whether a context starts with the tile passes.  Beside the sizes above they need, for nine tenths of the particles,
// boxes that fit LDS, and lists that hold the neighbours: what does not fit is searched for one particle at a time,
// from HBM.  A step by tiles / by variant 2 (us): boxes that do not fit, 64,000 particles (46 a cell) 625 / 512,
// 250,047 (46) 1,833 / 919, (104) 5,111 / 2,246; lists that do not, 1,000,000 (268 neighbours, 256 entries) 30,502 /
// 4,372, 4,492,125 (151, 128 entries) 141,144 / 10,523.
//
// Where both fit, by occupancy.  Up to 16 a cell they gain at any size (343,000 particles, 15.6 a cell, 423 / 552;
// 1,000,000, 14.7, 1,014 / 1,069; 4,492,125, 14.8, 4,097 / 4,343).  Above, lanes of a workgroup idle; with a kernel
// radius of the cell's side, or (r) of 0.84 of it, where less of that work finds neighbours:
//   16 to 20:    343,000 (17) 537 / 586, but 704,969 (17) 972 / 954, 2,000,376 (17) 2,694 / 2,324
//                r: 1,481,544 (17) 1,136 / 1,270, but 2,985,984 (19) 2,653 / 2,579
//   20 to 22.5:  1,000,000 (21) 1,278 / 1,396, but 2,000,376 (21) 2,645 / 2,546
//                r: 1,481,544 (21) 1,426 / 1,466, but 2,985,984 (20) 2,879 / 2,807
//   22.5 to 28:  704,969 (27) 1,007 / 1,251, 4,492,125 (27) 6,706 / 7,007
//   28 and more: 704,969 (30, 123 neighbours) 1,380 / 1,454, but 1,000,000 (30, 127) 2,200 / 1,995;
//                2,985,984 (32, 103) 4,489 / 4,747, r: (32) 3,835 / 4,379
inline bool start_on_tiles(const std::vector<SceneFill>& scenes, const TileShape& t) {
    double n = 0.0, cell = 0.0, over = 0.0, neighbours = 0.0;
    for (const SceneFill& f : scenes) {
        if (f.n == 0.0) continue;
        n += f.n;
        cell += f.occupancy * f.n;
        if ((t.x + 2) * (t.y + 2) * (t.z + 2) * f.occupancy * 1.05 > t.cap) over += f.n;
        if (f.neighbours > neighbours) neighbours = f.neighbours;
    }
    if (n < kTileMinParticles || n < (double)kTileMinPerScene * (double)scenes.size()) return false;
    if (over > 0.1 * n || neighbours * 1.1 > tile_list_cap((uint64_t)n)) return false;
    cell /= n;
    constexpr double kAny = 1e18;
    const bool narrow = neighbours <= 2.7 * cell;
    const double most = cell <= 16.0   ? kAny
                        : cell < 20.0  ? (narrow ? 2e6 : 4e5)
                        : cell < 22.5  ? (narrow ? 2e6 : 1.2e6)
                        : cell < 28.0  ? kAny
                                       : (neighbours <= 110.0 ? kAny : 8e5);
    return n <= most;
}

// Boxes with at most this many records per cell of the box and its halo are not staged: their particles' slots go to
// the list of sparse ones, which is searched directly.  A fluid that has spread over the cube, us a step of three
// contexts at once, with no such line / 1.33 / 2 / 3 / 4 records: 192,089 particles at step 4,000 140 / 98 / 97 / 98 /
// 103 (105 by the per-particle passes), a million at step 2,000 405 / 370 / 363 / 364 / 369 (467).  A block at its
// start has few thin boxes, in its skin, and a context that does not fill the chip waits for their particles: by 2 / 3
// (one context) 64,000 particles 73 / 100, 250,047 108 / 134, but 493,000 186 / 187, 704,969 270 / 272, a million 328 /
// 328.  A gas that fills the cube, 2 / 3 / by variant 2: a million, two a cell 706 / 587 / 640, three a cell 705 / 667
// / 689; 195,112, two a cell, 189 / 162 / 175; 64,000 121 / 111 / 100.
inline uint32_t sparse_records(uint64_t particles) { return particles >= 600000 ? 3u : 2u; }

// The tuner's candidates from the times t[lists][pass][variant] of the density and force pass: the fastest pair without
// neighbour lists, with them, and the last variant's (by tiles), whose passes run only with each other and form the
// same lists in both modes.  Which of them it is, whole steps decide: the tile passes' sort also forms their work list
// and tables (a million particles 20 us, 17.8 million 0.28 ms), and a pass timed alone finds its data in the caches.
// Left out are candidates too far behind for either (times in ms).
struct TuningPick {
    int density, update;
    bool lists;
};
inline std::vector<TuningPick> tuning_candidates(const std::vector<double> (&t)[2][2], bool tiles) {
    const int tile = (int)t[0][0].size() - 1;
    std::vector<TuningPick> all, out;
    std::vector<double> sum;
    for (int mode = 0; mode < 2; ++mode) {
        int best[2] = {0, 0};
        for (int pass = 0; pass < 2; ++pass)
            for (int v = 1; v < tile; ++v)
                if (t[mode][pass][v] < t[mode][pass][best[pass]]) best[pass] = v;
        all.push_back({best[0], best[1], mode == 1});
        sum.push_back(t[mode][0][best[0]] + t[mode][1][best[1]]);
    }
    if (tiles) {
        all.push_back({tile, tile, true});
        sum.push_back(fmin(t[0][0][tile], t[1][0][tile]) + fmin(t[0][1][tile], t[1][1][tile]));
    }
    double least = sum[0];
    for (double v : sum) least = fmin(least, v);
    for (size_t k = 0; k < all.size(); ++k)
        if (sum[k] <= 1.3 * least + 0.05) out.push_back(all[k]);
    return out;
}

}  // namespace wc
