// Chunk <-> brick maps of the coders that quantize inside the encoder and
// dequantize inside the decoder: direct_bricks_fit (z bands of a power of two)
// and rank_bricks_fit (the other fields of full bricks). Host+device so that CPU
// tests check them against the recursive octant rank (cpu/src/codec.cpp:96-107).
#pragma once

#include <cstdint>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define WZP_HD __host__ __device__ __forceinline__
#else
#define WZP_HD inline
#endif

namespace wz {

// The map of direct_bricks_fit written out for one kind of field, full 16^3
// bricks in pairs (no kernel uses it by itself): WZP chunk c, i.e. magnitudes
// [8192c, 8192c + 8192), is exactly bricks 2c and 2c+1 of the row-major brick
// grid (brick base = brick index * 4096), and the 32 ranks [32t, 32t + 32) of
// that chunk form one 4x4x2 sub-block: in a 16^3 brick the recursive rank has
// bits z3 y3 x3 z2 y2 x2 z1 y1 x1 z0 y0 x0 from most to least significant, so
// the low five bits are x0 y0 z0 x1 y1.
constexpr bool pair_bricks_fit(uint32_t nx, uint32_t ny, uint32_t nz, uint32_t bz) {
    return bz == 16 && nx % 32 == 0 && ny % 16 == 0 && nz % 16 == 0 && nx && ny && nz;
}

// Origin of the sub-block holding ranks [32t, 32t+32) of chunk c (t < 256).
WZP_HD void pair_subblock(uint32_t nx, uint32_t ny, uint32_t c, uint32_t t, uint32_t& x, uint32_t& y,
                          uint32_t& z) {
    const uint32_t nbx = nx / 16, nby = ny / 16;
    const uint32_t b = 2 * c + (t >> 7);
    const uint32_t xi = b % nbx, r = b / nbx, yi = r % nby, zi = r / nby;
    const uint32_t u = t & 127u;  // rank bits 5..11: z1 x2 y2 z2 x3 y3 z3
    x = 16 * xi + 4 * ((u >> 1) & 1u) + 8 * ((u >> 4) & 1u);
    y = 16 * yi + 4 * ((u >> 2) & 1u) + 8 * ((u >> 5) & 1u);
    z = 16 * zi + 2 * (u & 1u) + 4 * ((u >> 3) & 1u) + 8 * ((u >> 6) & 1u);
}

// Rank (0..31) inside the sub-block of offset (dx, dy, dz), dx, dy < 4, dz < 2.
WZP_HD constexpr uint32_t subblock_rank(uint32_t dx, uint32_t dy, uint32_t dz) {
    return (dx & 1u) | ((dy & 1u) << 1) | (dz << 2) | ((dx >> 1) << 3) | ((dy >> 1) << 4);
}

// The same for full bricks whose z band is a power of two up to 16 (nx, ny
// multiples of 16, nz of the band): a brick holds 256 bz packed
// positions and 32 divides its start, so the 32 positions of a thread are one
// sub-block of one brick whose place follows from the position's bits. From
// least to most significant the rank bits are, for bz = 16: x0 y0 z0 x1 y1 z1
// x2 y2 z2 x3 y3 z3; 8: x0 y0 x1 y1 z0 x2 y2 z1 x3 y3 z2; 4: x0 y0 x1 y1 x2 y2
// z0 x3 y3 z1; 2: x0 y0 x1 y1 x2 y2 x3 y3 z0; 1: the same without z0. The
// sub-block is 4 x 4 x 2 for bz >= 8 and 8 x 4 x 1 below: eight runs of four
// x-consecutive samples, run r at y offset r & 3 and, from r = 4 on, one
// plane or four samples further.
// `size`: bytes of a sample. Against the coders of rank_bricks_fit, which go
// through an LDS image of the chunk, floats gain (encoder / decoder: 256^3,
// band 8, 47 -> 36 / 46 -> 34 us; 384x384x64, band 2, 33 -> 25 / 29 -> 27;
// 128^3, band 8, 25 -> 15 / 30 -> 18). Doubles of a flat band do not: a
// thread's runs are 32-byte pieces of rows that its neighbours in the wave do
// not continue (256x256x128, band 8, encoder 28 -> 29, decoder 30 -> 38), so
// they stay there; cubes take this path for both (no rank table, and the pairs
// of planes share their lines).
constexpr bool direct_bricks_fit(uint32_t nx, uint32_t ny, uint32_t nz, uint32_t bz, uint32_t size) {
    return (bz == 16 || (size == 4 && (bz == 1 || bz == 2 || bz == 4 || bz == 8))) && nx % 16 == 0 && ny % 16 == 0 &&
           nz % bz == 0 && nx && ny && nz;
}
constexpr uint32_t log2_band(uint32_t bz) { return bz >= 16 ? 4 : bz >= 8 ? 3 : bz >= 4 ? 2 : bz >= 2 ? 1 : 0; }

// Origin of the sub-block of packed positions [8192 c + 32 t, + 32).
WZP_HD void direct_subblock(uint32_t nx, uint32_t ny, uint32_t lbz, uint32_t c, uint32_t t, uint32_t& x, uint32_t& y,
                            uint32_t& z) {
    const uint32_t p = 256 * c + t, b = p >> (3 + lbz), u = p & ((8u << lbz) - 1u);  // in units of 32
    const uint32_t nbx = nx / 16, nby = ny / 16;
    const uint32_t r = b / nbx, xi = b - r * nbx, zi = r / nby, yi = r - zi * nby;
    auto bit = [u](uint32_t k) { return (u >> k) & 1u; };
    if (lbz == 4) {
        x = 4 * bit(1) + 8 * bit(4);
        y = 4 * bit(2) + 8 * bit(5);
        z = 2 * bit(0) + 4 * bit(3) + 8 * bit(6);
    } else if (lbz == 3) {
        x = 4 * bit(0) + 8 * bit(3);
        y = 4 * bit(1) + 8 * bit(4);
        z = 2 * bit(2) + 4 * bit(5);
    } else if (lbz == 2) {
        x = 8 * bit(2);
        y = 4 * bit(0) + 8 * bit(3);
        z = bit(1) + 2 * bit(4);
    } else {
        x = 8 * bit(1);
        y = 4 * bit(0) + 8 * bit(2);
        z = bit(3);  // (u has no such bit for a band of 1)
    }
    x += 16 * xi;
    y += 16 * yi;
    z += zi << lbz;
}
// Rank (0..31) inside the sub-block of sample dx of run r; Cube: bz = 16.
template <bool Cube>
WZP_HD constexpr uint32_t direct_rank(uint32_t dx, uint32_t r) {
    return Cube ? subblock_rank(dx, r & 3u, r >> 2)
                : (dx & 1u) | ((r & 1u) << 1) | ((dx >> 1) << 2) | (((r >> 1) & 1u) << 3) | ((r >> 2) << 4);
}
// The same the other way round.
template <bool Cube>
WZP_HD constexpr void direct_place(uint32_t rank, uint32_t& dx, uint32_t& r) {
    auto bit = [rank](uint32_t k) { return (rank >> k) & 1u; };
    if (Cube) {
        dx = bit(0) | bit(3) << 1;
        r = bit(1) | bit(4) << 1 | bit(2) << 2;
    } else {
        dx = bit(0) | bit(2) << 1;
        r = bit(1) | bit(3) << 1 | bit(4) << 2;
    }
}

// Chunk <-> brick map of the other fields of full bricks (z bands that are no
// power of two, doubles of a band below 16): brick b of the row-major brick
// grid holds packed positions [bV, bV + V), V = 256 bz, in recursive
// octant rank order (one table of V ranks, the full brick's), and chunk c
// holds packed positions [8192c, 8192c + E), so the bricks of a chunk are
// consecutive (a chunk starts or ends inside a brick when V does not divide
// 8192). The (de)quantizing coders visit a chunk's bricks in row-major
// order, four x-consecutive samples at a time, and place each sample at its
// rank in the chunk.
constexpr bool rank_bricks_fit(uint32_t nx, uint32_t ny, uint32_t nz, uint32_t bz) {
    return bz >= 1 && bz <= 16 && nx % 16 == 0 && ny % 16 == 0 && nz % bz == 0 && nx && ny && nz;
}
// Bricks that can overlap one chunk (V = 256 at least, starting anywhere).
constexpr uint32_t kRankBricksMax = 8192 / 256 + 2;

}  // namespace wz
