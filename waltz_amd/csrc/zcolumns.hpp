// Z lifting of whole columns in registers: every Z level of the plane schedule
// in one pass (its Z phase), or one Z pass of a dyadic level, shared by the
// single-field and batched transforms.
#pragma once

#include "buffer.hpp"
#include "common.hpp"
#include "lifting.hpp"
#include "repair.hpp"
#include "windows.hpp"

namespace wz {

// A workgroup of four waves (more: zcol_threads) owns a row of 64 columns, all
// z; a wave takes one tile of the 64 columns at a time, a lane a column, so
// that a tile's rows, their mirrored places and its tests are wave-uniform
// (scalar): per sample only the lifting itself and its loads and stores reach
// the vector unit. The finest
// level reads (forward) or writes (inverse) the field and every high band
// goes between registers and the volume directly; only the low boxes between
// the levels pass through LDS, alternating between two buffers (box 1 in the
// first, ceil(nz/2) rows, box 2 in the second, box 3 in the first again), with
// one barrier per level. Tiles and arithmetic are those of the Z axis passes
// (lift_forward / lift_inverse folded), so the same bits; status: screen for
// non-finite samples the forward's input or the inverse's output. It reads and
// writes the field once, at 3.3-4.0 TB/s of the 5.1 that a copy reaches: the
// halo rows of the tiles and one level after the other. With every column
// staged in LDS and per-lane index arithmetic it was bound by vector issue:
// 500x500x100 float 108 -> 55 us (forward), 127 -> 61 us (inverse), 384x384x96
// double 70 -> 56 us, 73 -> 67 us.
//
// Repair (inverse, compress): the reconstruction is not written; each sample
// is compared with the original as its tile is lifted, and the native repair
// records and flag bits go out (one segment per workgroup, columns x nz slots).
// That drops a write and a read of the field and one launch: 384x384x96
// double 68 us, inverse and repair passes 67 + 47 before; where rows share flag
// words, which are set by atomics then, slower (500x500x100 float 88 us, 2.3 TB/s).

// Decides the samples v[j] (rows z + j of column x, row y) of a wave's tile
// against their originals, sets their flag bits and appends their records to
// segment `id`; false when a lane's sample cannot meet the bound. Wave masks
// as in the fused finest level: the rounded difference of the final value and
// the original settles the strict bound unless it is not below it.
template <class T, int Tile>
WZ_D bool zcol_repairs(const T (&v)[Tile], const T (&ref)[Tile], const WaveRepair<T>& rp, Dims full, uint32_t x,
                       uint32_t y, uint32_t z, bool in, uint32_t id, uint32_t* seg_fill) {
    const uint32_t lane = threadIdx.x & 63u;
    const unsigned long long in_m = __ballot(in);
    bool ok = true;
    unsigned long long masks[Tile];
    T err[Tile];
    uint32_t total = 0;
#pragma unroll
    for (int j = 0; j < Tile; ++j) {
        masks[j] = 0;
        err[j] = v[j] - ref[j];
        if (z + uint32_t(j) >= full.nz) continue;  // (wave-uniform)
        masks[j] = repair_mask<T>(v[j], ref[j], in, in_m, rp, &ok);
        total += uint32_t(__popcll(masks[j]));
    }
    uint32_t base = 0;
    if (total && lane == 0) base = atomicAdd(seg_fill, total);
    base = __builtin_amdgcn_readfirstlane(base);
    const uint32_t row_words = (full.nx & 31u) == 0;
    uint32_t at = uint32_t((uint64_t(z) * full.ny + y) * full.nx) + x;  // sample index of row z
    uint32_t* const index = rp.rep.index + uint64_t(id) * rp.rep.cap;
    T* const payload = static_cast<T*>(rp.rep.payload) + uint64_t(id) * rp.rep.cap;
#pragma unroll
    for (int j = 0; j < Tile; ++j) {
        if (z + uint32_t(j) >= full.nz) continue;
        const unsigned long long m = masks[j];
        const uint32_t first = at - lane;  // sample of lane 0
        if (row_words) {  // the row's 64 samples own whole words
            if (lane < 2 && x - lane + 32u * lane < full.nx)
                rp.rep.bitmap[(first >> 5) + lane] = uint32_t(m >> (32u * lane));
        } else if (m && lane < 3) {  // shared words of a cleared bitmap
            const uint32_t s = first & 31u;
            const unsigned long long lo = m << s;
            const uint32_t w = lane == 0   ? uint32_t(lo)
                               : lane == 1 ? uint32_t(lo >> 32)
                               : s         ? uint32_t(m >> (64u - s))
                                           : 0u;
            if (w) atomicOr(&rp.rep.bitmap[(first >> 5) + lane], w);
        }
        if ((m >> lane) & 1ull) {
            const uint32_t k = base + uint32_t(__popcll(m & ((1ull << lane) - 1ull)));
            index[k] = at;
            payload[k] = err[j];
        }
        base += uint32_t(__popcll(m));
        at += full.nx * full.ny;
    }
    return ok;
}

// What becomes of an inverse's finest samples besides the store: clipping to
// an output frame, a hole's fill value instead of them, a non-finite screen.
template <class T>
struct ZOutput {
    Dims clip;  // extents that are stored
    bool screen, hole;
    T fill;
};
// The source and destination volumes of a column pass (pitches in elements;
// nz planes of either, but only 16 of an inverse's destination, inside one
// 32-bit byte window; Wide: one plane of either) and the box lifted.
template <class T>
struct ZColumnsOf {
    const T* src;
    uint32_t spy, spz;
    T* dst;
    uint32_t dpy, dpz;
    Dims n;           // box: n.nx x n.ny columns of n.nz samples
    uint32_t levels;
};

// Row y, columns x0 .. x0 + 63 by one workgroup of `Threads` threads; `box0`,
// `box1`: zcol_lds_bytes of LDS. Returns whether this lane met nothing to flag
// (a non-finite sample of a screened pass, or an unmet bound). Wide: volumes
// past one window, every plane through its own (3370x3300x99 float, 4.4 GB:
// forward 2.2 ms, 4.0 TB/s). InPlace: src may be dst; the finest level's rows
// from `from` on wait in `held` (zcol_held_rows of LDS) until all are read.
template <class T, bool Inverse, bool Repair, bool Wide = false, bool InPlace = false, uint32_t Threads = kZThreads>
WZ_D bool zcol_columns(const ZColumnsOf<T>& a, uint32_t y, uint32_t x0, T* box0, T* box1, bool screen,
                       const ZOutput<T>& out, const WaveRepair<T>& rp, uint32_t id, uint32_t* seg_fill,
                       T* held = nullptr) {
    constexpr int Tile = sizeof(T) == 4 ? 16 : 8, P = Tile / 2 + 4;  // (the inverse's is part of the format)
    constexpr uint32_t W = Threads / 64, S = sizeof(T);
    static_assert(!(Repair && Wide), "the codec's fields fit one window");
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63u;
    const uint32_t x = x0 + lane;
    const bool in = x < a.n.nx;
    const uint32_t splane = a.spz * S, dplane = a.dpz * S;
    const uint32_t xc = in ? x : a.n.nx - 1u;
    const uint32_t scol = (y * a.spy + xc) * S, dcol = (y * a.dpy + xc) * S;
    const auto ws = window(a.src), wd = window(Repair ? rp.orig : a.dst);
    // plane z of the source / destination, `at`: its offset inside one window
    auto load = [&](uint32_t z, uint32_t at) {
        if constexpr (Wide) return buf_load<T>(window(a.src + uint64_t(z) * a.spz), scol);
        else return buf_load_at(T(0), ws, scol, at);
    };
    auto row = [&](uint32_t z) { return load(z, z * splane); };
    auto store = [&](T v, uint32_t z, uint32_t at) {
        if constexpr (Wide) buf_store(v, window(a.dst + uint64_t(z) * a.dpz), dcol);
        else buf_store_at(v, wd, dcol, at);
    };
    [[maybe_unused]] const uint32_t from = a.n.nz - zcol_held_rows(a.n.nz, a.levels);
    auto hold = [&](T v, uint32_t z) { held[(z - from) * kZColumns + lane] = v; };
    // the finest inverse store's lanes and rows
    const bool put = Inverse ? x < out.clip.nx && y < out.clip.ny : in;
    const int32_t rows = int32_t(Inverse ? out.clip.nz : a.n.nz);
    bool fin = true;
    for (uint32_t k = 0; k < a.levels; ++k) {
        const uint32_t l = Inverse ? a.levels - 1 - k : k;
        uint32_t m = a.n.nz;
        for (uint32_t i = 0; i < l; ++i) m = half_len(m);
        const int32_t n = int32_t(m), h = int32_t(half_len(m));
        const bool finest = l == 0, coarsest = l + 1 == a.levels;
        // this level's box (l >= 1) and the next coarser one
        T* const own = (l & 1u) ? box0 : box1;
        T* const low = (l & 1u) ? box1 : box0;
        for (uint32_t tile = wave; int32_t(tile) * Tile < n; tile += W) {
            T e[P], o[P];
            const int32_t k0 = int32_t(tile) * (Tile / 2) - 2;
            const bool inner = k0 >= 0 && 2 * (k0 + P) <= n;  // no mirrored position
            if constexpr (!Inverse) {
                if (finest) {
                    if (inner) {
                        uint32_t at = uint32_t(2 * k0) * splane;
#pragma unroll
                        for (int j = 0; j < P; ++j) {
                            e[j] = load(uint32_t(2 * (k0 + j)), at);
                            o[j] = load(uint32_t(2 * (k0 + j) + 1), at + splane);
                            at += 2 * splane;
                        }
                    } else {
#pragma unroll
                        for (int j = 0; j < P; ++j) {
                            e[j] = row(uint32_t(2 * pair_even(k0 + j, n)));
                            o[j] = row(uint32_t(2 * pair_odd(k0 + j, n) + 1));
                        }
                    }
                    if (screen) {
#pragma unroll
                        for (int j = 2; j < P - 2; ++j) fin = fin && finite_value(e[j]) && finite_value(o[j]);
                    }
                } else {
                    const T* b = own + lane;
#pragma unroll
                    for (int j = 0; j < P; ++j) {
                        e[j] = b[uint32_t(2 * pair_even(k0 + j, n)) * kZColumns];
                        o[j] = b[uint32_t(2 * pair_odd(k0 + j, n) + 1) * kZColumns];
                    }
                }
                lift_forward<T, P>(e, o);
                T* b = low + uint32_t(k0 + 2) * kZColumns + lane;
                uint32_t at = uint32_t(k0 + 2) * dplane, up = uint32_t(k0 + 2 + h) * dplane;
#pragma unroll
                for (int j = 2; j < P - 2; ++j) {
                    if (2 * (k0 + j) < n) {
                        if (!coarsest) b[uint32_t(j - 2) * kZColumns] = e[j];
                        else if (InPlace && finest) hold(e[j], uint32_t(k0 + j));
                        else if (in) store(e[j], uint32_t(k0 + j), at);
                    }
                    if (InPlace && finest) {
                        if (2 * (k0 + j) + 1 < n) hold(o[j], uint32_t(k0 + j + h));
                    } else if (2 * (k0 + j) + 1 < n && in) {
                        store(o[j], uint32_t(k0 + j + h), up);
                    }
                    at += dplane;
                    up += dplane;
                }
            } else {
                if (inner) {
                    uint32_t at = uint32_t(k0) * splane, up = uint32_t(k0 + h) * splane;
#pragma unroll
                    for (int j = 0; j < P; ++j) {
                        if (coarsest) e[j] = load(uint32_t(k0 + j), at);
                        o[j] = load(uint32_t(k0 + j + h), up);
                        at += splane;
                        up += splane;
                    }
                } else {
#pragma unroll
                    for (int j = 0; j < P; ++j) {
                        if (coarsest) e[j] = row(uint32_t(pair_even(k0 + j, n)));
                        o[j] = row(uint32_t(h + pair_odd(k0 + j, n)));
                    }
                }
                T ref[Repair ? Tile : 1];  // the tile's originals, in flight with its coefficients
                if constexpr (Repair) {
                    if (finest) {
                        uint32_t at = tile * uint32_t(Tile) * dplane;
#pragma unroll
                        for (int j = 0; j < Tile; ++j) {
                            ref[j] = buf_load_at_nt(T(0), wd, dcol, int32_t(tile) * Tile + j < n ? at : 0u);
                            at += dplane;
                        }
                    }
                }
                if (!coarsest) {
                    const T* b = low + lane;
#pragma unroll
                    for (int j = 0; j < P; ++j) e[j] = b[uint32_t(pair_even(k0 + j, n)) * kZColumns];
                }
                lift_inverse<T, P, true>(e, o);
                if constexpr (Repair) {
                    if (finest) {
                        T v[Tile];
#pragma unroll
                        for (int j = 0; j < Tile / 2; ++j) {
                            v[2 * j] = e[j + 2];
                            v[2 * j + 1] = o[j + 2];
                        }
                        const uint32_t z = tile * uint32_t(Tile);
                        fin = zcol_repairs<T, Tile>(v, ref, rp, a.n, x, y, z, in, id, seg_fill) && fin;
                        continue;
                    }
                }
                if (!finest) {
                    T* b = own + uint32_t(2 * (k0 + 2)) * kZColumns + lane;
#pragma unroll
                    for (int j = 2; j < P - 2; ++j) {
                        if (2 * (k0 + j) < n) b[uint32_t(2 * (j - 2)) * kZColumns] = e[j];
                        if (2 * (k0 + j) + 1 < n) b[uint32_t(2 * (j - 2) + 1) * kZColumns] = o[j];
                    }
                    continue;
                }
                // (a tile's rows only inside one window: frames may be large)
                const uint32_t z0 = tile * uint32_t(Tile);
                const auto wt = window(a.dst + uint64_t(z0) * a.dpz);
                uint32_t at = 0;
#pragma unroll
                for (int j = 2; j < P - 2; ++j) {
#pragma unroll
                    for (int b = 0; b < 2; ++b) {
                        if (2 * (k0 + j) + b < rows) {
                            const T v = out.hole ? out.fill : b ? o[j] : e[j];
                            const uint32_t z = uint32_t(2 * (k0 + j) + b);
                            if (InPlace && z >= from) {
                                hold(v, z);
                            } else if (put) {
                                if constexpr (Wide) store(v, z, 0u);
                                else buf_store_at(v, wt, dcol, at);
                            }
                            if (out.screen) fin = fin && (finite_value(v) || !put || out.hole);
                        }
                        at += dplane;
                    }
                }
            }
        }
        __syncthreads();
        if constexpr (InPlace) {
            if (finest)
                for (uint32_t z = from + wave; z < a.n.nz; z += W)
                    if (in) store(held[(z - from) * kZColumns + lane], z, z * dplane);
        }
    }
    return fin;
}

// One Z level of a box, one wave per item: a tile of 64 columns, columns
// counted row by row so that narrow boxes fill the lanes. Items: z_items().
template <class T>
WZ_HD uint32_t z_items(Dims n) {
    constexpr uint32_t Tile = sizeof(T) == 4 ? 16 : 8;
    return ((n.nx * n.ny + 63) / 64) * ((n.nz + Tile - 1) / Tile);
}
template <class T, bool Inverse>
WZ_D void z_tile(const T* src, T* dst, uint32_t py, uint32_t pz, Dims box, uint32_t item) {
    constexpr int Tile = sizeof(T) == 4 ? 16 : 8, P = Tile / 2 + 4;
    constexpr uint32_t S = sizeof(T);
    const int32_t n = int32_t(box.nz), h = int32_t(half_len(box.nz));
    const uint32_t columns = box.nx * box.ny, blocks = (columns + 63) / 64;
    const uint32_t tile = item / blocks, c = (item - tile * blocks) * 64u + (threadIdx.x & 63u);
    const bool in = c < columns;
    const uint32_t cc = in ? c : 0u, y = cc / box.nx;
    const uint32_t col = (y * py + (cc - y * box.nx)) * S, plane = pz * S;
    const auto ws = window(src), wd = window(dst);
    const int32_t k0 = int32_t(tile) * (Tile / 2) - 2;
    T e[P], o[P];
#pragma unroll
    for (int j = 0; j < P; ++j) {
        const uint32_t ie = uint32_t(pair_even(k0 + j, n)), io = uint32_t(pair_odd(k0 + j, n));
        e[j] = buf_load_at(T(0), ws, col, (Inverse ? ie : 2 * ie) * plane);
        o[j] = buf_load_at(T(0), ws, col, (Inverse ? uint32_t(h) + io : 2 * io + 1) * plane);
    }
    if constexpr (Inverse) lift_inverse<T, P, true>(e, o);
    else lift_forward<T, P>(e, o);
    if (!in) return;
#pragma unroll
    for (int j = 2; j < P - 2; ++j) {
        const uint32_t k = uint32_t(k0 + j);
        if (2 * int32_t(k) < n) buf_store_at(e[j], wd, col, (Inverse ? 2 * k : k) * plane);
        if (2 * int32_t(k) + 1 < n) buf_store_at(o[j], wd, col, (Inverse ? 2 * k + 1 : uint32_t(h) + k) * plane);
    }
}

}  // namespace wz
