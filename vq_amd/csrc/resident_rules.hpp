// Which reconstructions take their table into LDS, by groups of columns that blockIdx.y numbers: rules on sizes alone,
// without HIP, so that a CPU test can go through them.
#pragma once
#include <algorithm>
#include <cstdint>

namespace vq {

constexpr int64_t kMaxGridY = 65535;  // workgroups in the second dimension of a grid

// Column blocks per group of k_decode_resident; 0: the gather (k_decode_gather).  Kernel times behind an assignment of
// as many rows, gather -> table.
// A centroid of one 16-byte piece of the output: the table in LDS once the codebook is more than the vector
// cache holds, from 2^19 pieces on.  f16 blocks of 8: 200,000 x 12, k = 256 11.9 -> 9.6 us, 1M x 16, k = 256 91 -> 54; geometric
// means 1.04 below 2^19 pieces, 0.96 (8 MB written), 0.85 (16 to 64 MB).  f32 blocks of 4: 1.1-1.2 with tables up to 32 KB, 0.97 at
// 64 KB, 0.86 at 128.
// More pieces, which the gather reads as one run of bytes: the gather, until the rows (240 MB of f32) leave
// nothing of the output in the memory-side cache.  Stores that go to memory want the table's long runs, others do not:
// f16 100,000 x 12 blocks of 32 1.05-1.3, from 60M elements on 0.65-0.88 (1M x 8 of 16, k = 256 71 -> 54); f32 1.05-1.3, then
// 0.74-0.92 (1M x 16 of 8, k = 256 123 -> 104).
// Where the blocks' tables exceed LDS a group's share of every row has to be whole 64-byte halves of lines, the stores
// pass the caches: 1M x 16, k = 1024 (two groups) 75 -> 50, 300,000 x 32, k = 512 47 -> 31, 66,000 x 64, k = 2048 (64-byte shares) 32.6 ->
// 22.3; with shares that end inside: 1M x 10, k = 1024 48 -> 121, 300,000 x 17, k = 2048, f32 30 -> 129.
// The last group may be short and its runs long: their places are counted in 32 bits.
inline int decode_resident_blocks(bool f16, int64_t n, int m, int sd, int k) {
    const int64_t line = (int64_t)sd * (f16 ? 2 : 4), pieces = line / 16, block = k * line, room = 128 * 1024;
    if (line % 16 != 0 || block > room || n * m < (1 << 16)) return 0;
    const bool beyond = n * m * sd >= 60'000'000;
    int64_t G = m;
    if (block * m <= room) {
        if (!beyond && (pieces > 1 || n * m < (1 << 19) || block * m < (f16 ? 8 : 64) * 1024)) return 0;
    } else {
        G = room / block;
        if (G * line >= 128) G = G * line / 128 * 128 / line;
        if (G < 1 || G * line % 64 != 0 || m * line % 64 != 0 || n * m < (1 << 20) || (pieces > 1 && !beyond)) return 0;
    }
    const int64_t groups = (m + G - 1) / G, last = m - (groups - 1) * G;
    const int64_t rows = std::min<int64_t>(n, std::max<int64_t>(1, (f16 ? 4096 : 8192) / (last * pieces)));
    if (groups > kMaxGridY || rows * m * pieces >= (1LL << 32)) return 0;
    return (int)G;
}

// Whether binary16 rows of blocks that fill no 16-byte pieces are made from a table in LDS (k_decode_flat; else
// k_decode_units): the table is filled once per workgroup, so from 64 values of the output per value of the table on, and from
// sizes on where a launch is not most of the time.  Alone, units -> table: 372,160 x 21 blocks of 15, k = 33 147 -> 59 us (4.0 TB/s),
// 755,499 x 8 of 7, k = 216 59 -> 25, 322,755 x 49 of 7, k = 227 (156 KB) 156 -> 67, 122,321 x 55 of 2, k = 189 23.5 -> 10.5, 300,000 x 10 of 12,
// k = 256 22 -> 17, x 16 of 4 18.8 -> 9.4, 20,000 x 60 of 5, k = 256 (79 values per value) 12.3 -> 11.5, 6,000 x 30 of 15, k = 30 6.4 -> 6.0;
// below the lines 6,404 x 17 of 7, k = 98 4.9 -> 6.1, 20,000 x 16 of 6, k = 256 5.1 -> 5.9, 8,000 x 50 of 3, k = 256 5.2 -> 7.7.
constexpr int kDecodeFlatLds = 160 * 1024;  // the largest table, bytes
inline bool decode_flat_resident(int64_t n, int64_t m, int64_t sd, int64_t k) {
    constexpr int64_t most = kDecodeFlatLds / 2;
    if (m > most || sd > most || m * sd * k > most) return false;
    const int64_t total = n * m * sd;
    return total >= (sd % 4 == 0 ? 5'000'000 : 2'500'000) && total >= 64 * (m * sd * k);
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
