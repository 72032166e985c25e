// Which reconstructions take their table into LDS, by groups of columns that blockIdx.y numbers: rules on sizes alone,
// without HIP, so that a CPU test can go through them.
#pragma once
#include <algorithm>
#include <cstdint>

namespace vq {

constexpr int64_t kMaxGridY = 65535;  // workgroups in the second dimension of a grid

// Column blocks per group of k_decode_resident; 0: the gather.  The table of all blocks within 128 KB, or, where there
// are enough rows for the groups' tables, a group of blocks whose pieces of a row fill whole lines, or half of one.
// A short last group has the longest runs, up to 8192 rows of m blocks: its places are counted in 32 bits.
inline int decode_resident_blocks(bool f16, int64_t n, int m, int sd, int k) {
    const int64_t block = (int64_t)k * sd * (f16 ? 2 : 4), line = (int64_t)sd * (f16 ? 2 : 4);
    if (sd % (f16 ? 8 : 4) != 0 || block > 128 * 1024 || n * m < (1 << 16) || (int64_t)m * sd >= (1 << 24)) return 0;
    int64_t G = m;
    if (block * m > 128 * 1024) {
        G = 128 * 1024 / block;
        if (G * line >= 128) G = G * line / 128 * 128 / line;
        if (G < 1 || G * line < 64 || n * m < (1 << 20)) return 0;
    }
    const int64_t groups = (m + G - 1) / G, last = m - (groups - 1) * G, pieces = line / 16;
    const int64_t rows = std::min<int64_t>(n, std::max<int64_t>(1, (f16 ? 4096 : 8192) / (last * pieces)));
    if (groups > kMaxGridY || rows * m * pieces >= (1LL << 32)) return 0;
    return (int)G;
}

}  // namespace vq
