// Which volumes the kernels with 32-bit byte offsets take. Host code without
// HIP, so that a CPU test checks the rules against the offsets.
#pragma once

#include <cstdint>

namespace wz {

// Whether `rows` rows of pitch `pitch` elements of `width` bytes stay below
// 4 GiB less 1 MiB (the level kernels' 32-bit byte offsets within a plane,
// with room above the plane for the offset that masks a lane off).
inline bool fused_plane_fits(uint64_t pitch, uint64_t rows, uint64_t width) {
    return pitch * rows * width <= (uint64_t(1) << 32) - (uint64_t(1) << 20);
}

// Column passes (zcolumns.hpp): LDS rows of 64 columns for the low boxes between
// the levels, ceil(nz/2) and ceil(nz/4) of them.
constexpr uint32_t kZColumns = 64;
constexpr uint32_t zcol_lds_rows(uint32_t nz, unsigned levels) {
    const uint32_t n1 = nz - nz / 2;
    return levels < 2 ? 0u : levels > 2 ? n1 + (n1 - n1 / 2) : n1;
}
// In place: the finest level's results that would overwrite rows it still reads
// (the high half, of a single level both) wait in LDS behind those.
constexpr uint32_t zcol_held_rows(uint32_t nz, unsigned levels) { return levels > 1 ? nz / 2 : nz; }
constexpr uint64_t zcol_lds_bytes(uint32_t nz, unsigned levels, unsigned width, bool in_place = false) {
    return (uint64_t(zcol_lds_rows(nz, levels)) + (in_place ? zcol_held_rows(nz, levels) : 0u)) * kZColumns * width;
}
// 64 KiB of LDS: nz up to 340 (float) or 170 (double) whatever the levels, in
// place up to 204 or 102
constexpr bool zcol_lds_fits(uint32_t nz, unsigned width) { return zcol_lds_bytes(nz, 5, width) <= 65536; }
constexpr bool zcol_place_fits(uint32_t nz, unsigned levels, unsigned width) {
    return zcol_lds_bytes(nz, levels, width, true) <= 65536;
}
// Threads of a workgroup of columns, by the workgroups of the launch and their
// LDS. Where a CU gets no second workgroup, a row of columns is a chain of tiles
// per wave and lasts the longer the fewer its waves are (260x60x9 float, z first:
// compress 131 us with 4 waves, 114 with 8, 107 with 16; 200x200x64 float forward
// 19.3, 16.1, 15.1). Beyond that four are enough (100x2000x64 float inverse 29.5,
// 35.9, 68.3), except in place where LDS holds the workgroups of a CU to two or
// three (100x2000x64 double, 64 KiB: 59.6, 51.2, 68.7; 99x3300x3370, 5.7, 4.8 ms;
// but 60x3300x3370, 38 KiB: 2.5, 2.6).
constexpr uint32_t kZThreads = 256, kZThreadsPlace = 512, kZThreadsMost = 1024;
constexpr uint32_t zcol_threads(uint64_t workgroups, bool in_place, uint64_t lds) {
    return workgroups <= 256 ? kZThreadsMost : in_place && lds > 49152 ? kZThreadsPlace : kZThreads;
}
// Whether every one of `levels` levels lifts lines of at least two samples. One
// sample is its own even and odd neighbour: kernels that address the two halves
// of a line apart would read past it.
inline bool lines_fit(uint32_t n, unsigned levels) {
    for (unsigned l = 0; l < levels; ++l, n -= n / 2)
        if (n < 2) return false;
    return true;
}
// Whether the Z phase of an nx x ny x nz volume runs as columns, ...
inline bool zcol_fits(uint32_t nx, uint32_t ny, uint32_t nz, unsigned levels, unsigned width) {
    return zcol_lds_fits(nz, width) && lines_fit(nz, levels) && fused_plane_fits(nx, ny, width);
}
// ... and whether it has to address every plane through a window of its own:
// one window (of 2^32 - 1 bytes, no lane masked off by its offset) holds every
// field of the codec, but not every volume of the transforms.
inline bool zcol_wide(uint32_t nx, uint32_t ny, uint32_t nz, unsigned width) {
    return uint64_t(nx) * ny > 0xFFFFFFFFull / width / nz;
}

}  // namespace wz
