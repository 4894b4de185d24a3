// Rules of windows.hpp against the byte offsets the kernels form: a volume
// that is not `wide` has every offset of its samples below 2^32 - 1 (one
// buffer window), a volume that runs as columns at all has every offset of one
// plane there.
#include <cstdio>
#include <initializer_list>

#include "../waltz_amd/csrc/windows.hpp"

using namespace wz;

static int failures = 0;

static void check(uint32_t nx, uint32_t ny, uint32_t nz, unsigned width, bool fits, bool wide) {
    const uint64_t plane = uint64_t(nx) * ny * width, volume = plane * nz;
    const bool one = volume <= 0xFFFFFFFFull;  // the end of the last sample
    bool ok = zcol_fits(nx, ny, nz, 0, width) == fits;
    if (fits) {
        ok = ok && zcol_wide(nx, ny, nz, width) == wide && wide == !one;
        ok = ok && plane <= 0xFFFFFFFFull;
        // what a pass with one window would address: no offset may wrap
        if (!wide) ok = ok && uint64_t(uint32_t(volume - width)) == volume - width;
    }
    if (!ok) {
        std::printf("%ux%ux%u width %u: fits %d wide %d\n", nz, ny, nx, width, zcol_fits(nx, ny, nz, 0, width),
                    zcol_wide(nx, ny, nz, width));
        ++failures;
    }
}

int main() {
    check(500, 500, 100, 4, true, false);
    check(384, 384, 96, 8, true, false);
    // both sides of one window
    check(3500, 3500, 87, 4, true, false);
    check(3500, 3500, 88, 4, true, true);
    check(3500, 3500, 100, 4, true, true);
    check(4096, 4096, 96, 4, true, true);
    check(32768, 2048, 16, 4, true, true);   // 2^32 bytes
    check(65520, 16384, 1, 4, true, false);  // 2^32 - 2^20: the largest plane
    check(2730, 2048, 96, 8, true, false);   // 2^32 - 2^21
    check(2731, 2048, 96, 8, true, true);
    // the codec's largest fields stay in one window (n <= (2^32 - 1) / width)
    check(1073741823u / 9, 1, 9, 4, true, false);
    check(536870911u / 9, 1, 9, 8, true, false);
    // planes past a window
    check(65521, 16384, 9, 4, false, true);
    check(32768, 32760, 9, 4, true, true);
    check(32768, 32768, 9, 4, false, true);
    check(32768, 16384, 9, 8, false, true);
    check(65536, 65535, 9, 8, false, true);
    // LDS
    for (unsigned width : {4u, 8u}) {
        const uint32_t top = width == 4 ? 340 : 170;
        check(64, 64, top, width, true, false);
        check(64, 64, top + 1, width, false, false);
        if (zcol_lds_bytes(top, 5, width) > 65536 || zcol_lds_bytes(top + 1, 5, width) <= 65536) {
            std::printf("LDS limit, width %u\n", width);
            ++failures;
        }
    }
    // lines of one sample, at the first level and later
    const struct { uint32_t n; unsigned levels; bool fit; } lines[] = {
        {1, 0, true}, {1, 1, false}, {2, 1, true}, {2, 2, false}, {3, 2, true}, {3, 3, false}, {9, 4, true}, {9, 5, false},
        {16, 4, true}, {16, 5, false}, {17, 5, true}, {340, 5, true}};
    for (const auto& k : lines) {
        bool ok = lines_fit(k.n, k.levels) == k.fit && zcol_fits(64, 64, k.n, k.levels, 4) == k.fit;
        // what a pass addresses: the halves of a line of m samples start at 0 and ceil(m / 2), both inside it
        uint32_t m = k.n;
        for (unsigned l = 0; k.fit && l < k.levels; ++l, m -= m / 2) ok = ok && m - m / 2 < m;
        if (!ok) {
            std::printf("lines of %u, %u levels\n", k.n, k.levels);
            ++failures;
        }
    }
    return failures != 0;
}
