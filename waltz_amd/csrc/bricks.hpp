// Morton bricks of a coefficient volume (cpu/src/codec.cpp:96-150): brick
// enumeration and packed base, and the quantization of one brick, shared by
// the single-field and batched pipelines.
#pragma once

#include "common.hpp"
#include "launch.hpp"

namespace wz {

struct Brick {
    uint32_t x0, y0, z0, bx, by, bz, shape;
    uint64_t base;
};

// Position (x, y, z) in brick k of its local row-major index i: shifts for
// bricks full in x and y (all but the edge ones), integer division otherwise.
WZ_D void brick_xyz(const Brick& k, uint32_t i, uint32_t& x, uint32_t& y, uint32_t& z) {
    if (k.bx == 16 && k.by == 16) {
        x = i & 15u;
        y = (i >> 4) & 15u;
        z = i >> 8;
    } else {
        const uint32_t r = i / k.bx;
        x = i - r * k.bx;
        y = r % k.by;
        z = r / k.by;
    }
}

WZ_D Brick brick_of(const BrickGeometry& g, uint32_t b) {
    Brick k;
    const uint32_t bxi = b % g.nbx, r = b / g.nbx, byi = r % g.nby, bzi = r / g.nby;
    k.x0 = bxi * 16;
    k.y0 = byi * 16;
    k.z0 = bzi * g.bz;
    k.bx = min(16u, g.d.nx - k.x0);
    k.by = min(16u, g.d.ny - k.y0);
    k.bz = min(g.bz, g.d.nz - k.z0);
    k.shape = unsigned(k.bx != 16) | (unsigned(k.by != 16) << 1) | (unsigned(k.bz != g.bz) << 2);
    k.base = uint64_t(k.z0) * g.d.nx * g.d.ny + uint64_t(k.y0) * g.d.nx * k.bz + uint64_t(k.x0) * k.by * k.bz;
    return k;
}

// Samples a workgroup of the separate quantization pass takes at most, and the
// bricks that may be (full bricks hold 256 bz samples).
constexpr uint32_t kGroupSamples = 8192, kGroupBricks = 32;
WZ_HD uint32_t group_bricks(uint32_t bz) { return bz >= 32 ? 1u : 32u / bz; }

// Bricks [first, first + count) of a field (one workgroup of 256 threads, count
// <= group_bricks): coefficients quantized, written back dequantized inside
// `box` only, u16 magnitudes at their packed ranks (`rank`: the eight edge
// shapes' tables), sign bits, q-outliers appended.
//
// Consecutive bricks are consecutive in the packed order, so the group's
// magnitudes are gathered in LDS and leave as whole 16-byte words, as its sign
// bits leave as 32-bit words; a thread takes four neighbours of a brick at a
// time and has the loads of four such quads in flight. What bounds it is
// memory latency, hence several bricks per workgroup: a workgroup per brick,
// with every magnitude a 2-byte store, took 118 us on 500x500x100 floats (z
// band 4: 1024 samples a brick), this takes 51 (also without writing
// the coefficients back, which the inverse levels quantize as they load).
template <class T>
WZ_D void quantize_group(T* __restrict__ coeff, const BrickGeometry& g, T q, T inv, const uint16_t* __restrict__ rank,
                         uint16_t* __restrict__ mag, uint32_t* __restrict__ sign, const SideList& qo,
                         uint32_t* __restrict__ status, uint32_t first, uint32_t count, Dims box) {
    __shared__ Brick kb[kGroupBricks];
    __shared__ __attribute__((aligned(16))) uint16_t mags[kGroupSamples + 8];
    __shared__ uint32_t bits[kGroupSamples / 32 + 1];
    const uint32_t t = threadIdx.x;
    if (t < count) kb[t] = brick_of(g, first + t);
    for (uint32_t w = t; w < kGroupSamples / 32 + 1; w += 256) bits[w] = 0;
    __syncthreads();
    const Brick& kl = kb[count - 1];
    const uint64_t base0 = kb[0].base;
    const uint32_t total = uint32_t(kl.base - base0) + kl.bx * kl.by * kl.bz;
    const uint32_t shift = uint32_t(base0 & 31u);
    const uint32_t lead = uint32_t(reinterpret_cast<uintptr_t>(mag + base0) / 2) & 7u;
    const uint32_t quads = 64u * g.bz;  // of a full brick
    bool bad = false;
    constexpr uint32_t kBurst = 4;
    for (uint32_t f0 = 0; f0 < count * quads; f0 += kBurst * 256u) {
        T v[kBurst][4];
        uint16_t rv[kBurst][4];
        uint32_t jb[kBurst], li[kBurst], held[kBurst], over = 0;
        auto place = [&](uint32_t u, uint32_t k) -> uint64_t {
            const Brick& b = kb[jb[u]];
            uint32_t x, y, z;
            brick_xyz(b, li[u] + k, x, y, z);
            return (uint64_t(b.z0 + z) * g.d.ny + (b.y0 + y)) * g.d.nx + b.x0 + x;
        };
#pragma unroll
        for (uint32_t u = 0; u < kBurst; ++u) {
            // (a wave's 64 quads are one brick's)
            const uint32_t f = f0 + u * 256u + t, w = __builtin_amdgcn_readfirstlane(f >> 6);
            const uint32_t j = w / g.bz;
            const bool in = j < count;
            jb[u] = in ? j : 0u;
            const Brick& b = kb[jb[u]];
            const uint32_t vol = b.bx * b.by * b.bz;
            li[u] = 4u * (f - j * quads);
            held[u] = in && li[u] < vol ? min(4u, vol - li[u]) : 0u;
            if (!held[u]) li[u] = 0;
            __builtin_memcpy(rv[u], rank + b.shape * 8192u + li[u], 8);
            if (b.bx == 16) {
                __builtin_memcpy(v[u], coeff + place(u, 0), 4 * sizeof(T));
            } else {
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k) v[u][k] = coeff[place(u, k < held[u] ? k : 0u)];
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < kBurst; ++u) {
            const Brick& b = kb[jb[u]];
            const uint32_t rel = uint32_t(b.base - base0);
            T d[4];
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) {
                if (k >= held[u]) continue;
                // cpu/src/quantize_avx2.cpp:45-62: finite and |scaled| < 2^63
                // (one compare: false for NaN and infinities), llrint, INT32
                // saturation
                const T scaled = v[u][k] * inv;
                bad = bad || !(abs_t(scaled) < T(9223372036854775808.0));
                const T rounded = rint_t(scaled);
                const uint32_t m = quantum_count(abs_t(rounded)), p = rel + rv[u][k];
                d[k] = m ? T(rounded < T(0) ? -int32_t(m) : int32_t(m)) * q : T(0);
                mags[lead + p] = uint16_t(m > 65535u ? 65535u : m);
                if (rounded < T(0)) atomicOr(&bits[(p + shift) >> 5], 1u << ((p + shift) & 31u));
                over |= uint32_t(m > 65535u) << (4 * u + k);
            }
            if (!held[u] || b.x0 >= box.nx || b.y0 >= box.ny || b.z0 >= box.nz) continue;
            uint32_t x, y, z;
            brick_xyz(b, li[u], x, y, z);
            if (b.bx == 16 && b.x0 + x + 4 <= box.nx) {
                if (b.y0 + y < box.ny && b.z0 + z < box.nz) __builtin_memcpy(coeff + place(u, 0), d, 4 * sizeof(T));
            } else {
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k) {
                    if (k >= held[u]) continue;
                    brick_xyz(b, li[u] + k, x, y, z);
                    if (b.x0 + x < box.nx && b.y0 + y < box.ny && b.z0 + z < box.nz) coeff[place(u, k)] = d[k];
                }
            }
        }
        append_qoutliers<4 * kBurst>(
            qo, over, [&](int i) { return uint32_t(place(uint32_t(i) / 4, uint32_t(i) % 4)); },
            [&](int i) { return quantum_count(abs_t(rint_t(v[i / 4][i % 4] * inv))); });
    }
    if (bad) atomicOr(status, uint32_t(kQuantDomain));
    __syncthreads();
    // whole 16-byte words of magnitudes; the first and the last may be shared
    uint16_t* const dst = mag + base0 - lead;
    for (uint32_t w = 8 * t; w < lead + total; w += 8 * 256u) {
        if (w >= lead && w + 8 <= lead + total) {
            *reinterpret_cast<uint4*>(dst + w) = *reinterpret_cast<const uint4*>(mags + w);
        } else {
            for (uint32_t k = max(w, lead); k < min(w + 8, lead + total); ++k) dst[k] = mags[k];
        }
    }
    // The group's bits are global bits [base0, base0 + total); LDS word w maps
    // to global word base0 / 32 + w. The first and last words may be shared
    // with neighbours.
    const uint32_t words = (shift + total + 31) >> 5;
    const uint64_t w0 = base0 >> 5;
    for (uint32_t w = t; w < words; w += 256) {
        const uint32_t b = bits[w];
        if (w == 0 || w == words - 1) {
            if (b) atomicOr(&sign[w0 + w], b);
        } else {
            sign[w0 + w] = b;
        }
    }
}

}  // namespace wz
