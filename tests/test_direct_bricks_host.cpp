// Every sample of a field of full bricks lands, through direct_subblock and
// direct_rank, on the magnitude position the brick layout gives it (base of
// brick + recursive octant rank), for every z band of a power of two and brick
// counts that leave the last chunk partial.
#include <cstdint>
#include <cstdio>
#include <vector>

#include "../waltz_amd/csrc/bits.hpp"
#include "../waltz_amd/csrc/pairbrick.hpp"

using namespace wz;

static uint32_t octant_rank(uint32_t x, uint32_t y, uint32_t z, uint32_t nx, uint32_t ny, uint32_t nz) {
    uint32_t rank = 0;
    while (nx > 1 || ny > 1 || nz > 1) {
        const uint32_t lx = nx - nx / 2, ly = ny - ny / 2, lz = nz - nz / 2;
        const uint32_t sz = z < lz ? lz : nz - lz, sy = y < ly ? ly : ny - ly, sx = x < lx ? lx : nx - lx;
        if (z >= lz) { rank += lz * ny * nx; z -= lz; }
        if (y >= ly) { rank += sz * ly * nx; y -= ly; }
        if (x >= lx) { rank += sz * sy * lx; x -= lx; }
        nx = sx;
        ny = sy;
        nz = sz;
    }
    return rank;
}

template <bool Cube>
static int check(uint32_t nx, uint32_t ny, uint32_t nz, uint32_t bz) {
    if (!direct_bricks_fit(nx, ny, nz, bz, 4)) return 1;
    const uint32_t n = nx * ny * nz, lbz = log2_band(bz), up = lbz >= 3 ? nx * ny : 4;
    int bad = 0;
    std::vector<uint8_t> seen(n, 0);
    for (uint32_t p = 0; p < n; p += 32) {
        uint32_t X, Y, Z;
        direct_subblock(nx, ny, lbz, p / 8192, p % 8192 / 32, X, Y, Z);
        for (uint32_t r = 0; r < 8; ++r)
            for (uint32_t dx = 0; dx < 4; ++dx) {
                const uint32_t at = (Z * ny + Y) * nx + X + (r & 3) * nx + (r >> 2) * up + dx;
                if (at >= n) { ++bad; continue; }
                const uint32_t x = at % nx, y = at / nx % ny, z = at / nx / ny;
                const uint32_t x0 = x / 16 * 16, y0 = y / 16 * 16, z0 = z / bz * bz;
                const uint32_t base = z0 * nx * ny + y0 * nx * bz + x0 * 16 * bz;
                bad += base + octant_rank(x - x0, y - y0, z - z0, 16, 16, bz) != p + direct_rank<Cube>(dx, r);
                ++seen[at];
            }
    }
    for (uint8_t v : seen) bad += v != 1;
    return bad;
}

// The sample a rank belongs to, and the nonzero mask of a pair of bit planes.
template <bool Cube>
static int check_places() {
    int bad = 0;
    for (uint32_t i = 0; i < 32; ++i) {
        uint32_t dx, r;
        direct_place<Cube>(i, dx, r);
        bad += dx > 3 || r > 7 || direct_rank<Cube>(dx, r) != i;
    }
    return bad;
}
static int check_nonzero() {
    int bad = 0;
    uint32_t x = 12345;
    for (int it = 0; it < 20000; ++it) {
        uint32_t m[32], planes[16], nz = 0;
        for (int i = 0; i < 32; ++i) {
            x = x * 1664525u + 1013904223u;
            m[i] = it < 32 ? uint32_t(i == it) << (it & 15) : (x >> 30) ? 0u : (x >> 8 & 0xFFFFu) >> (x >> 4 & 15u);
            nz |= uint32_t(m[i] != 0) << i;
        }
        bit2_forward_pair(m, planes);
        bad += pair_nonzero(planes) != nz;
    }
    return bad;
}

int main() {
    int bad = check_places<true>() + check_places<false>() + check_nonzero();
    bad += check<true>(48, 32, 32, 16) + check<true>(16, 16, 16, 16);
    for (uint32_t bz : {1u, 2u, 4u, 8u})
        bad += check<false>(48, 32, 3 * bz, bz) + check<false>(16, 16, bz, bz) + check<false>(112, 48, 5 * bz, bz);
    bad += direct_bricks_fit(48, 40, 32, 16, 4) || direct_bricks_fit(48, 48, 36, 12, 4) || direct_bricks_fit(40, 48, 32, 4, 4) ||
           direct_bricks_fit(48, 48, 34, 4, 4);
    std::printf("bad = %d\n", bad);
    return bad != 0;
}
