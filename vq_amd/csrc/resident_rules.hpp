// Which reconstructions take their table into LDS, by groups of columns that blockIdx.y numbers: rules on sizes alone,
// without HIP, so that a CPU test can go through them.
#pragma once
#include <algorithm>
#include <cstdint>

namespace vq {

constexpr int64_t kMaxGridY = 65535;  // workgroups in the second dimension of a grid

// Column blocks per group of k_decode_resident; 0: the gather (k_decode_gather).
// The table in LDS pays where a centroid is one 16-byte piece of the output and the codebook is more than the vector
// cache holds, from 2^19 pieces on.  Gather -> table, f16 blocks of 8, output not in a cache: 1M x 16, k = 256 67 -> 50 us, 200,000 x 12
// 12.0 -> 9.5, 1M x 10 41 -> 34; geometric means by table size 1.03 (1-4 KB), 0.97 (8 KB), 0.92 (16 KB), 0.84 (32), 0.80 (64-128); below
// 2^19 pieces 1.08 (5.4 -> 5.8 us).  f32 blocks of 4: 1.1-1.2 up to 32 KB (200,000 x 12, k = 256 9.4 -> 12.3), 0.97 at 64 KB, 0.86
// at 128.
// Where the blocks' tables exceed LDS a group's share of every row has to be whole 64-byte halves of lines, the stores
// pass the caches: 1M x 16, k = 1024 (two groups) 75 -> 50, 300,000 x 32, k = 512 47 -> 31, 66,000 x 64, k = 2048 (64-byte shares) 32.6 ->
// 22.3; with shares that end inside: 1M x 10, k = 1024 48 -> 121, 300,000 x 17, k = 2048, f32 30 -> 129.
// Centroids of more than one piece are read by the gather as one run of bytes: 1M x 4 blocks of 32, k = 1024
// 41 -> 51, 110,000 x 12 of 32, k = 16 14.6 -> 20.5 (geometric means 1.04-1.7 by width).
// The last group may be short and its runs long: their places are counted in 32 bits.
inline int decode_resident_blocks(bool f16, int64_t n, int m, int sd, int k) {
    const int64_t table = (int64_t)k * 16 * m, room = 128 * 1024;
    if (sd != (f16 ? 8 : 4) || n * m < (1 << 19) || table < (f16 ? 8 : 64) * 1024) return 0;
    int64_t G = m;
    if (table > room) {
        G = room / ((int64_t)k * 16);
        G = G >= 8 ? G / 8 * 8 : G / 4 * 4;
        if (G == 0 || m % 4 != 0 || n * m < (1 << 20)) return 0;
    }
    const int64_t groups = (m + G - 1) / G, last = m - (groups - 1) * G;
    const int64_t rows = std::min<int64_t>(n, std::max<int64_t>(1, (f16 ? 4096 : 8192) / last));
    if (groups > kMaxGridY || rows * m >= (1LL << 32)) return 0;
    return (int)G;
}

// Columns per group of k_rvq_recon_resident; 0: the gather.  The stages' table within 128 KB, 32 columns or more, or 16.
// Where groups share rows that are not whole halves of lines, from four stages on: gather -> resident of 256 centroids
// 200,000 x 72, two stages 14.9 -> 15.0 us, 400,000 33.6 -> 42.8, 400,000 x 104 38 -> 50; four stages 200,000 x 136 39 -> 31, 400,000 60 -> 63,
// 200,000 x 264 65 -> 56; six 49 -> 37 (200,000 x 136); geometric means over seven widths 1.08, 0.87, 0.83.
inline int rvq_recon_columns(int64_t n, int stages, int k, int dim) {
    if (dim % 8 != 0 || stages < 1 || (int64_t)stages * k > 2048) return 0;
    const int most = 32 * 1024 / (stages * k), fit = most < 32 ? 16 : most / 32 * 32;
    if (fit >= dim) return dim;
    const int64_t groups = (dim + fit - 1) / fit, last = dim - (groups - 1) * fit;
    const int64_t rows = std::min<int64_t>(n, std::max<int64_t>(1, 2048 / (last / 8)));  // of a run of the last group
    if (groups > kMaxGridY || rows * (dim / 8) >= (1LL << 32)) return 0;  // places in a run: 32 bits
    return dim % 32 != 0 && stages < 4 ? 0 : fit;
}

}  // namespace vq
