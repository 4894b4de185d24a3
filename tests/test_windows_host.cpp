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
    bool ok = zcol_fits(nx, ny, nz, width) == fits;
    if (fits) {
        ok = ok && zcol_wide(nx, ny, nz, width) == wide && wide == !one;
        ok = ok && plane <= 0xFFFFFFFFull;
        // what a pass with one window would address: no offset may wrap
        if (!wide) ok = ok && uint64_t(uint32_t(volume - width)) == volume - width;
    }
    if (!ok) {
        std::printf("%ux%ux%u width %u: fits %d wide %d\n", nz, ny, nx, width, zcol_fits(nx, ny, nz, width),
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
    return failures != 0;
}
