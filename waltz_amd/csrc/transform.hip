// CDF 9/7 lifting passes for gfx950.
//
// The plane schedule is one pass over all Z levels (zcolumns.hpp) and one launch
// per XY level (xystrip.hpp), its coarse planes in one (planetail.hpp); a dyadic
// level is one fused launch (fused.hip), or a Z axis pass and one XY launch, the
// coarsest boxes in one workgroup. What none of these fits is left to the axis
// passes:
//
// One launch lifts one axis of the active low box [0,act.nx)x[0,act.ny)x[0,act.nz)
// of a full row-major volume (x fastest), out of place: src -> dst, both with
// the full volume's strides. Each thread owns one canonical tile of one line:
// it loads P = Tile/2+4 (even, odd) sample pairs into registers (reflected at
// the axis ends), runs the lifting steps there and writes Tile outputs.
//
// Tiles follow the reference CPU halo schedule (cpu/src/transform.cpp:113-179,
// 377-456). Forward tiles and the inverse X tile are bit-neutral; the inverse
// Y tile (8) and Z tile (16 for f32, 8 for f64) are part of the format because
// the two endpoint sums of a Y/Z tile are contracted into one fma each
// (cpu/src/transform.cpp:115-129).
//
// Y and Z lines map consecutive lanes to consecutive x, so every register load
// is a fully coalesced 256 B (f32) / 512 B (f64) wave access; X lines map lanes
// to consecutive tiles of one row (overlapping 64 B windows served from L1).
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <map>
#include <mutex>
#include <string>
#include <tuple>
#include <type_traits>

#include "buffer.hpp"
#include "common.hpp"
#include "fused.hpp"
#include "launch.hpp"
#include "lifting.hpp"
#include "planetail.hpp"
#include "profile.hpp"
#include "xystrip.hpp"
#include "zcolumns.hpp"

namespace wz {

// Axis: 0 = X, 1 = Y, 2 = Z.
template <class T, bool Inverse, int Axis, int Tile>
__global__ void __launch_bounds__(256) axis_pass(const T* __restrict__ src, T* __restrict__ dst, Dims full,
                                                 Dims act, uint32_t ntiles, uint32_t total,
                                                 uint32_t* __restrict__ status) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= total) return;
    uint32_t x = 0, y = 0, z = 0, t;
    if constexpr (Axis == 0) {
        t = i % ntiles;
        const uint32_t r = i / ntiles;
        y = r % act.ny;
        z = r / act.ny;
    } else if constexpr (Axis == 1) {
        x = i % act.nx;
        const uint32_t r = i / act.nx;
        t = r % ntiles;
        z = r / ntiles;
    } else {
        x = i % act.nx;
        const uint32_t r = i / act.nx;
        y = r % act.ny;
        t = r / act.ny;
    }
    const uint64_t plane = uint64_t(full.nx) * full.ny;
    const uint32_t n = Axis == 0 ? act.nx : Axis == 1 ? act.ny : act.nz;
    const uint64_t stride = Axis == 0 ? 1u : Axis == 1 ? uint64_t(full.nx) : plane;
    const uint64_t base = uint64_t(z) * plane + uint64_t(y) * full.nx + x;
    lift_tile<T, Inverse, Axis, Tile>(src, base, stride, dst, base, stride, n, t, status);
}

// Two consecutive in-plane passes (X then Y, or Y then X) of a small box in
// one launch: one workgroup per z plane stages the plane in LDS, runs the
// first pass LDS to LDS and the second LDS to dst. The same tile lifting as
// axis_pass, so the same bits.
template <class T, bool Inverse, int A0, int A1, uint32_t kPlaneMax>
__global__ void __launch_bounds__(256) plane_pair_pass(const T* __restrict__ src, T* __restrict__ dst, Dims full,
                                                       Dims act) {
    __shared__ T P0[kPlaneMax], P1[kPlaneMax];  // kPlaneMax: samples of a staged plane
    const uint32_t z = blockIdx.x, t = threadIdx.x;
    const uint64_t plane = uint64_t(full.nx) * full.ny, zb = uint64_t(z) * plane;
    const uint32_t cells = act.nx * act.ny;
    for (uint32_t i = t; i < cells; i += 256u) P0[i] = src[zb + uint64_t(i / act.nx) * full.nx + i % act.nx];
    __syncthreads();
    auto pass = [&](auto axis_c, const T* s, uint64_t sbase, uint64_t spitch, T* d, uint64_t dbase, uint64_t dpitch) {
        constexpr int A = decltype(axis_c)::value;
        const uint32_t n = A == 0 ? act.nx : act.ny, lines = A == 0 ? act.ny : act.nx;
        const uint32_t ntiles = (n + 7) / 8;
        for (uint32_t i = t; i < lines * ntiles; i += 256u) {
            const uint32_t tile = i % ntiles, line = i / ntiles;
            // X: line y, stride 1; Y: line x, stride = the row pitch
            const uint64_t so = A == 0 ? uint64_t(line) * spitch : line, ss = A == 0 ? 1u : spitch;
            const uint64_t dof = A == 0 ? uint64_t(line) * dpitch : line, ds = A == 0 ? 1u : dpitch;
            lift_tile<T, Inverse, A, 8>(s, sbase + so, ss, d, dbase + dof, ds, n, tile, nullptr);
        }
    };
    pass(std::integral_constant<int, A0>{}, P0, 0, act.nx, P1, 0, act.nx);
    __syncthreads();
    pass(std::integral_constant<int, A1>{}, P1, 0, act.nx, dst, zb, full.nx);
}

// Box `act` of a full-pitch volume, quantized and dequantized (the value a
// coefficient holds after quantization), to a compact array of pitch act.nx.
template <class T>
__global__ void __launch_bounds__(256) box_requant(const T* __restrict__ src, T* __restrict__ dst, Dims full, Dims act,
                                                   uint32_t total, T q, T inv) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= total) return;
    const uint32_t x = i % act.nx, r = i / act.nx, y = r % act.ny, z = r / act.ny;
    dst[i] = requantize<T>(src[(uint64_t(z) * full.ny + y) * full.nx + x], q, inv);
}

template <class T>
__global__ void __launch_bounds__(256) box_copy(const T* __restrict__ src, T* __restrict__ dst, Dims full, Dims act,
                                                uint32_t total) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= total) return;
    const uint32_t x = i % act.nx, r = i / act.nx, y = r % act.ny, z = r / act.ny;
    const uint64_t at = (uint64_t(z) * full.ny + y) * full.nx + x;
    dst[at] = src[at];
}

namespace {
Dims shrink(Dims d, bool xy, bool z) {
    if (xy) { d.nx = half_len(d.nx); d.ny = half_len(d.ny); }
    if (z) d.nz = half_len(d.nz);
    return d;
}

template <class T, bool Inverse, int Axis, int Tile>
void launch_axis(const T* src, T* dst, Dims full, Dims act, uint32_t* status, hipStream_t stream) {
    const uint32_t n = Axis == 0 ? act.nx : Axis == 1 ? act.ny : act.nz;
    const uint32_t ntiles = (n + Tile - 1) / Tile;
    const uint64_t lines = uint64_t(act.nx) * act.ny * act.nz / n;
    const uint64_t total = lines * ntiles;
    if (total == 0) return;
    check_launch_size(total);
    hipLaunchKernelGGL((axis_pass<T, Inverse, Axis, Tile>), dim3(uint32_t((total + 255) / 256)), dim3(256), 0, stream,
                       src, dst, full, act, ntiles, uint32_t(total), status);
}

// The line tile is free for forward passes and the inverse X pass (it only
// decides how a line is cut among threads; every tile recomputes its halo);
// the inverse Y and Z tiles are the canonical ones.
template <class T, bool Inverse, int Axis>
void launch_axis_tile(const T* src, T* dst, Dims full, Dims act, uint32_t tile, uint32_t* status, hipStream_t s) {
    if (tile == 32) launch_axis<T, Inverse, Axis, 32>(src, dst, full, act, status, s);
    else if (tile == 16) launch_axis<T, Inverse, Axis, 16>(src, dst, full, act, status, s);
    else launch_axis<T, Inverse, Axis, 8>(src, dst, full, act, status, s);
}

template <class T, bool Inverse>
void axis(const T* src, T* dst, Dims full, Dims act, int axis, const uint32_t* tiles, uint32_t* status,
          hipStream_t s) {
    constexpr int ZTileInv = sizeof(T) == 4 ? 16 : 8;
    if (axis == 0) launch_axis_tile<T, Inverse, 0>(src, dst, full, act, tiles[0], status, s);
    else if (Inverse && axis == 1) launch_axis<T, Inverse, 1, 8>(src, dst, full, act, status, s);
    else if (axis == 1) launch_axis_tile<T, Inverse, 1>(src, dst, full, act, tiles[1], status, s);
    else if (Inverse) launch_axis<T, Inverse, 2, ZTileInv>(src, dst, full, act, status, s);
    else launch_axis_tile<T, Inverse, 2>(src, dst, full, act, tiles[2], status, s);
}

template <class T, bool Inverse>
bool xy_pair(const T* src, T* dst, Dims full, Dims act, int a0, uint32_t* status, hipStream_t s);

// X and Y passes of a box in one launch: planes up to `limit` samples (tuned:
// 1024 or 4096, 0 = none) staged whole in LDS by one workgroup, larger ones
// and screened ones (status: the forward's input or the inverse's output) as
// strips.
template <class T, bool Inverse>
bool plane_pair(const T* src, T* dst, Dims full, Dims act, int a0, int a1, uint32_t limit, uint32_t* status,
                hipStream_t s) {
    const uint64_t cells = uint64_t(act.nx) * act.ny;
    if (act.nz == 0 || a0 + a1 != 1) return false;
    if (cells > limit || status) return xy_pair<T, Inverse>(src, dst, full, act, a0, status, s);
    if (cells <= 1024) {
        if (a0 == 0)
            hipLaunchKernelGGL((plane_pair_pass<T, Inverse, 0, 1, 1024>), dim3(act.nz), dim3(256), 0, s, src, dst,
                               full, act);
        else
            hipLaunchKernelGGL((plane_pair_pass<T, Inverse, 1, 0, 1024>), dim3(act.nz), dim3(256), 0, s, src, dst,
                               full, act);
    } else {
        if (a0 == 0)
            hipLaunchKernelGGL((plane_pair_pass<T, Inverse, 0, 1, 4096>), dim3(act.nz), dim3(256), 0, s, src, dst,
                               full, act);
        else
            hipLaunchKernelGGL((plane_pair_pass<T, Inverse, 1, 0, 4096>), dim3(act.nz), dim3(256), 0, s, src, dst,
                               full, act);
    }
    return true;
}

bool zcol_fits(Dims n, unsigned levels, unsigned width) { return wz::zcol_fits(n.nx, n.ny, n.nz, levels, width); }

template <class T, bool Inverse, bool Repair, bool Wide, bool InPlace, uint32_t Threads>
__global__ void __launch_bounds__(Threads) zcol_levels_kernel(ZColumnsOf<T> a, uint32_t* __restrict__ status,
                                                                WaveRepair<T> rp) {
    static_assert(Inverse || !Repair, "repairs follow the inverse");
    __shared__ uint32_t seg_fill;  // repair entries of this workgroup
    extern __shared__ __attribute__((aligned(16))) uint8_t zlds[];
    T* const box0 = reinterpret_cast<T*>(zlds);
    T* const box1 = box0 + uint64_t(half_len(a.n.nz)) * kZColumns;
    const uint32_t xb = (a.n.nx + kZColumns - 1) / kZColumns;
    // consecutive column rows go to one XCD (workgroups are dealt to the eight
    // in turn): rows are no multiple of a cache line in general, and
    // neighbours share the lines at their ends
    const uint32_t total = xb * a.n.ny, per = (total + 7) / 8;
    const uint32_t id = (blockIdx.x & 7u) * per + (blockIdx.x >> 3);
    if (id >= total) return;
    if constexpr (Repair) {
        if (threadIdx.x == 0) seg_fill = 0;
        __syncthreads();
    }
    const bool screen = status && !Repair;
    T* const held = InPlace ? box0 + zcol_lds_rows(a.n.nz, a.levels) * kZColumns : nullptr;
    const bool fin = zcol_columns<T, Inverse, Repair, Wide, InPlace, Threads>(
        a, id / xb, (id % xb) * kZColumns, box0, box1, screen, ZOutput<T>{a.n, screen, false, T(0)}, rp, id, &seg_fill,
        held);
    if (status && __ballot(!fin) && (threadIdx.x & 63u) == 0)
        atomicOr(status, uint32_t(Repair ? kRepairBound : Inverse ? kNonFiniteOutput : kNonFiniteInput));
    if constexpr (Repair) {
        if (threadIdx.x == 0) rp.rep.count[id] = seg_fill;
    }
}

template <class T, bool Inverse>
void zcol_levels(const T* src, T* dst, Dims full, unsigned levels, uint32_t* status, hipStream_t s,
                 const WaveRepair<T>* repair = nullptr) {
    const bool place = src == dst;
    if (!zcol_fits(full, levels, sizeof(T)) || levels < 1 || levels > 5 ||
        (place && (repair || !zcol_place_fits(full.nz, levels, sizeof(T)))))
        throw std::logic_error("Z phase does not fit LDS");
    const bool wide = zcol_wide(full.nx, full.ny, full.nz, sizeof(T));
    const uint64_t total = uint64_t(full.ny) * ((full.nx + kZColumns - 1) / kZColumns);
    const uint64_t blocks = 8 * ((total + 7) / 8);
    const dim3 grid{uint32_t(blocks)};
    const uint32_t lds = uint32_t(zcol_lds_bytes(full.nz, levels, sizeof(T), place));
    const ZColumnsOf<T> a{src, full.nx, full.nx * full.ny, dst, full.nx, full.nx * full.ny, full, uint32_t(levels)};
    if (repair && (wide || repair->rep.segments != total ||
                   repair->rep.cap < uint64_t(std::min(full.nx, kZColumns)) * full.nz))
        throw std::logic_error("repair segments do not match the Z phase's launch");
    const uint32_t threads = zcol_threads(total, place, lds);
    check_launch_size(blocks * threads);
    auto launch = [&](auto repair_c, auto wide_c, auto place_c) {
        constexpr bool R = decltype(repair_c)::value, W = decltype(wide_c)::value, P = decltype(place_c)::value;
        const WaveRepair<T> rp = R ? *repair : WaveRepair<T>{};
        auto run = [&](auto threads_c) {
            constexpr uint32_t N = decltype(threads_c)::value;
            hipLaunchKernelGGL((zcol_levels_kernel<T, Inverse, R, W, P, N>), grid, dim3(N), lds, s, a, status, rp);
        };
        if constexpr (!W) {  // (volumes past a window have more workgroups)
            if (threads == kZThreadsMost) return run(std::integral_constant<uint32_t, kZThreadsMost>{});
        }
        if constexpr (P) {
            if (threads == kZThreadsPlace) return run(std::integral_constant<uint32_t, kZThreadsPlace>{});
        }
        run(std::integral_constant<uint32_t, kZThreads>{});
    };
    constexpr std::true_type yes{};
    constexpr std::false_type no{};
    if constexpr (Inverse) {
        if (repair) return launch(yes, no, no);
    }
    if (wide && place) launch(no, yes, yes);
    else if (wide) launch(no, yes, no);
    else if (place) launch(no, no, yes);
    else launch(no, no, no);
}

template <class T, bool Requant, bool Screen>
__global__ void __launch_bounds__(kStripThreads) xy_inverse_kernel(XYInverse<T> a, StripPlan p, uint32_t* status) {
    uint32_t item;
    if (!strip_of_wave(p, item)) return;
    if constexpr (Screen) {
        StripOutput<T> out{a.n, false, T(0)};
        strip_inverse<T, Requant>(a, p, item, out);
        if (__ballot(!out.finite) && (threadIdx.x & 63u) == 0) atomicOr(status, uint32_t(kNonFiniteOutput));
    } else {
        strip_inverse<T, Requant>(a, p, item, StripStore<T>{});
    }
}
template <class T, bool Wide>
__global__ void __launch_bounds__(kStripThreads) xy_forward_kernel(XYForward<T> a, StripPlan p) {
    uint32_t item;
    if (strip_of_wave(p, item)) strip_forward<T, false, Wide>(a, p, item);
}
// screen: flag non-finite results
template <class T>
void xy_inverse(const XYInverse<T>& a, hipStream_t s, uint32_t* screen = nullptr) {
    const StripPlan p = strip_plan(a.n, strips_pack(std::max({a.hpz, a.lpz, a.opz}), sizeof(T)));
    const dim3 grid(strip_blocks(p)), block(kStripThreads);
    if (a.q > T(0) && screen) throw std::logic_error("requantizing levels are not screened");
    if (a.q > T(0)) hipLaunchKernelGGL((xy_inverse_kernel<T, true, false>), grid, block, 0, s, a, p, screen);
    else if (screen) hipLaunchKernelGGL((xy_inverse_kernel<T, false, true>), grid, block, 0, s, a, p, screen);
    else hipLaunchKernelGGL((xy_inverse_kernel<T, false, false>), grid, block, 0, s, a, p, screen);
}
template <class T>
void xy_forward(const XYForward<T>& a, hipStream_t s) {
    const StripPlan p = strip_plan(a.n, strips_pack(std::max({a.hpz, a.lpz, a.spz}), sizeof(T)));
    const dim3 grid(strip_blocks(p)), block(kStripThreads);
    if (fused_plane_fits(std::max({a.hpy, a.lpy, a.spy}), a.n.ny, sizeof(T)))
        hipLaunchKernelGGL((xy_forward_kernel<T, false>), grid, block, 0, s, a, p);
    else
        hipLaunchKernelGGL((xy_forward_kernel<T, true>), grid, block, 0, s, a, p);
}

// The finest level of a dyadic field (its Z pass done, in `src`) with the
// native repairs detected instead of the reconstruction stored.
template <class T>
__global__ void __launch_bounds__(kStripThreads) xy_repair_kernel(XYInverse<T> a, StripPlan p, WaveRepair<T> r,
                                                                  uint32_t* status) {
    uint32_t item;
    if (!strip_of_wave(p, item)) return;
    StripRepair<T> out{r};
    strip_inverse<T, false>(a, p, item, out);
    if (__ballot(!out.ok) && (threadIdx.x & 63u) == 0) atomicOr(status, uint32_t(kRepairBound));
}
template <class T>
XYInverse<T> repair_level(const T* src, Dims full, const WaveRepair<T>& r) {
    const uint64_t py = full.nx, pz = uint64_t(full.nx) * full.ny;
    return XYInverse<T>{src, py, pz, src, py, pz, const_cast<T*>(r.orig), py, pz, full, T(0), T(0), 0u};
}
template <class T>
StripPlan repair_plan(Dims full) {
    return strip_plan(full, strips_pack(uint64_t(full.nx) * full.ny, sizeof(T)));
}
template <class T>
void xy_repair(const T* src, Dims full, const WaveRepair<T>& r, uint32_t* status, hipStream_t s) {
    const StripPlan p = repair_plan<T>(full);
    if (r.rep.segments != p.items() || r.rep.cap < strip_repair_cap(p))
        throw std::logic_error("repair segments do not match the finest level's launch");
    StageClock clock("inverse_L0_repairs", s);
    hipLaunchKernelGGL((xy_repair_kernel<T>), dim3(strip_blocks(p)), dim3(kStripThreads), 0, s,
                       repair_level(src, full, r), p, r, status);
}

// The coarsest dyadic levels in one launch: boxes of at most kTailSamples are
// too small to be worth a launch per pass (about 5 us each; a level of 12x16x24
// takes 7 us here instead of 10). A box of 32^3 would take one CU 11 us per
// level, more than its two launches. One workgroup of 16 waves runs every
// pass of these levels, Z tiles and strips dealt to its waves, with a barrier
// between passes; the box goes through the scratch volume and L2 as before.
constexpr uint32_t kTailSamples = 8192, kTailWaves = 16;
template <class T>
struct Tail {
    T* home;  // coefficient volume and scratch, both at the field's pitches
    T* tmp;
    uint64_t py, pz;
    const T* first;  // forward: where the finest box lies (home, or the input)
    T* last;         // inverse: where the finest box goes (home, or the output)
    uint32_t levels;
    Dims n[5];          // finest first
    StripPlan plan[5];
    uint32_t* status;   // screen for non-finite samples, or unmet bounds
};
template <class T>
__global__ void __launch_bounds__(64 * kTailWaves) tail_forward_kernel(Tail<T> a) {
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (uint32_t l = 0; l < a.levels; ++l) {
        const XYForward<T> xy{l ? a.home : a.first, a.py, a.pz, a.tmp, a.py, a.pz, a.tmp, a.py, a.pz, a.n[l],
                              l ? nullptr : a.status};
        for (uint32_t i = wave; i < a.plan[l].items(); i += kTailWaves) strip_forward<T>(xy, a.plan[l], i);
        __syncthreads();
        for (uint32_t i = wave; i < z_items<T>(a.n[l]); i += kTailWaves)
            z_tile<T, false>(a.tmp, a.home, uint32_t(a.py), uint32_t(a.pz), a.n[l], i);
        __syncthreads();
    }
}
enum TailOut : int { kTailStore = 0, kTailScreen = 1, kTailRepair = 2 };
template <class T, int Out>
__global__ void __launch_bounds__(64 * kTailWaves) tail_inverse_kernel(Tail<T> a, WaveRepair<T> r) {
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int l = int(a.levels) - 1; l >= 0; --l) {
        for (uint32_t i = wave; i < z_items<T>(a.n[l]); i += kTailWaves)
            z_tile<T, true>(a.home, a.tmp, uint32_t(a.py), uint32_t(a.pz), a.n[l], i);
        __syncthreads();
        XYInverse<T> xy{a.tmp, a.py, a.pz, a.tmp, a.py, a.pz, l ? a.home : a.last, a.py, a.pz, a.n[l], T(0), T(0), 0u};
        if (Out != kTailStore && l == 0) {
            for (uint32_t i = wave; i < a.plan[0].items(); i += kTailWaves) {
                if constexpr (Out == kTailScreen) {
                    StripOutput<T> out{a.n[0], false, T(0)};
                    strip_inverse<T, false>(xy, a.plan[0], i, out);
                    if (__ballot(!out.finite) && (threadIdx.x & 63u) == 0)
                        atomicOr(a.status, uint32_t(kNonFiniteOutput));
                } else {
                    xy.out = const_cast<T*>(r.orig);
                    StripRepair<T> out{r};
                    strip_inverse<T, false>(xy, a.plan[0], i, out);
                    if (__ballot(!out.ok) && (threadIdx.x & 63u) == 0) atomicOr(a.status, uint32_t(kRepairBound));
                }
            }
        } else {
            for (uint32_t i = wave; i < a.plan[l].items(); i += kTailWaves)
                strip_inverse<T, false>(xy, a.plan[l], i, StripStore<T>{});
        }
        __syncthreads();
    }
}

// First level of the tail of a dyadic field whose levels below `from` run
// otherwise (lxy: none).
unsigned tail_level(Dims full, unsigned lxy, unsigned from, unsigned width) {
    Dims n = full;
    for (unsigned l = 0; l < lxy; ++l) {
        if (l >= from && uint64_t(n.nx) * n.ny * n.nz <= kTailSamples &&
            strips_fit(n, full.nx, full.ny, lxy - l, width) && lines_fit(n.nz, lxy - l))
            return l;
        n = shrink(n, true, true);
    }
    return lxy;
}
template <class T>
Tail<T> make_tail(T* home, T* tmp, Dims full, unsigned level, unsigned lxy) {
    Tail<T> t{};
    t.home = home;
    t.tmp = tmp;
    t.py = full.nx;
    t.pz = uint64_t(full.nx) * full.ny;
    t.first = home;
    t.last = home;
    t.levels = lxy - level;
    Dims n = full;
    for (unsigned l = 0; l < lxy; ++l) {
        if (l >= level) {
            t.n[l - level] = n;
            t.plan[l - level] = strip_plan(n, strips_pack(t.pz, sizeof(T)), kTailWaves, 16);
        }
        n = shrink(n, true, true);
    }
    return t;
}
template <class T>
void tail_forward(const Tail<T>& t, hipStream_t s) {
    StageClock clock("forward_tail", s);
    hipLaunchKernelGGL((tail_forward_kernel<T>), dim3(1), dim3(64 * kTailWaves), 0, s, t);
}
// `repair` (the finest box is the field): records instead of the store; the
// field's plan, whose items are the record segments.
template <class T>
void tail_inverse(Tail<T> t, Dims full, const WaveRepair<T>* repair, hipStream_t s) {
    StageClock clock("inverse_tail", s);
    const dim3 block(64 * kTailWaves);
    if (repair) {
        t.plan[0] = repair_plan<T>(full);
        if (repair->rep.segments != t.plan[0].items() || repair->rep.cap < strip_repair_cap(t.plan[0]))
            throw std::logic_error("repair segments do not match the finest level's launch");
        hipLaunchKernelGGL((tail_inverse_kernel<T, kTailRepair>), dim3(1), block, 0, s, t, *repair);
    } else if (t.status) {
        hipLaunchKernelGGL((tail_inverse_kernel<T, kTailScreen>), dim3(1), block, 0, s, t, WaveRepair<T>{});
    } else {
        hipLaunchKernelGGL((tail_inverse_kernel<T, kTailStore>), dim3(1), block, 0, s, t, WaveRepair<T>{});
    }
}

// The X and Y passes of box `act` (in full-pitched arrays, src != dst) as one
// launch, in the order the strips lift (forward Y then X, inverse X then Y);
// false for the other order and for boxes that strips do not take.
template <class T, bool Inverse>
bool xy_pair(const T* src, T* dst, Dims full, Dims act, int a0, uint32_t* status, hipStream_t s) {
    const uint64_t py = full.nx, pz = uint64_t(full.nx) * full.ny;
    if (!strips_fit(act, full.nx, full.ny, 1, sizeof(T))) return false;
    if constexpr (Inverse) {
        if (a0 != 0) return false;
        xy_inverse<T>(XYInverse<T>{src, py, pz, src, py, pz, dst, py, pz, act, T(0), T(0), 0u}, s, status);
    } else {
        if (a0 != 1) return false;
        xy_forward<T>(XYForward<T>{src, py, pz, dst, py, pz, dst, py, pz, act, status}, s);
    }
    return true;
}

template <class T>
void copy_box(const T* src, T* dst, Dims full, Dims act, hipStream_t s) {
    const uint64_t total = uint64_t(act.nx) * act.ny * act.nz;
    if (!total) return;
    check_launch_size(total);
    hipLaunchKernelGGL((box_copy<T>), dim3(uint32_t((total + 255) / 256)), dim3(256), 0, s, src, dst, full, act,
                       uint32_t(total));
}

// The source of the Z phase: `src`, or a copy of it in `scratch` where the
// phase ends in `src` itself and does not fit in place (one more pass over the
// volume, against two per level for axis passes).
template <class T>
const T* z_source(const T* src, const T* dst, T* scratch, Dims full, unsigned levels, hipStream_t s) {
    if (src != dst || zcol_place_fits(full.nz, levels, sizeof(T))) return src;
    hip_check(hipMemcpyAsync(scratch, src, uint64_t(full.nx) * full.ny * full.nz * sizeof(T), hipMemcpyDeviceToDevice,
                             s),
              "copy");
    return scratch;
}

// Runs a sequence of axis passes on one box: data starts in `home` (or in
// `first_src` for the very first pass), every pass is out of place, and the
// box ends in `home` (or in `last_dst` for the very last pass).
template <class T, bool Inverse>
struct Passes {
    T* home;
    T* tmp[2];
    const T* first_src;
    T* last_dst;
    uint32_t* status;
    hipStream_t s;
    Tuning tune;  // tiles and LDS pair limit of the per-axis passes
    bool first = true;
    unsigned base = 0;  // level number of the box's level 0 (stage names)
    // inverse: where non-finite samples of the last level's result are flagged
    // (null: not asked); `screened` when its last launch did
    uint32_t* out_status = nullptr;
    // inverse: the last level's result is compared with originals instead of
    // stored (out_status takes unmet bounds)
    const WaveRepair<T>* repair = nullptr;
    bool screened = false;

    // Passes: src -> tmp0 -> tmp1 -> ... -> final. A single pass whose source
    // is already `home` goes through tmp0 and is copied back.
    void level(Dims full, Dims act, const int* axes, int count, bool last_level, unsigned index) {
        static const char* fwd[] = {"forward_L0", "forward_L1", "forward_L2", "forward_L3", "forward_L4"};
        static const char* inv[] = {"inverse_L0", "inverse_L1", "inverse_L2", "inverse_L3", "inverse_L4"};
        StageClock clock(Inverse ? inv[index + base] : fwd[index + base], s);
        const T* src = first ? first_src : home;
        T* final_dst = last_level && last_dst ? last_dst : home;
        for (int k = 0; k < count; ++k) {
            uint32_t* const screen = first && k == 0 ? status : nullptr;
            // two in-plane passes: one launch
            const bool pair = k + 1 < count && axes[k] != 2 && axes[k + 1] != 2;
            const int last = pair ? k + 1 : k;
            T* const other = src == tmp[0] ? tmp[1] : tmp[0];  // never the source
            T* dst = last == count - 1 ? final_dst : other;
            if (dst == src) dst = other;  // in place at the end: through scratch, copied back below
            uint32_t* const out = Inverse && last_level && last == count - 1 ? out_status : nullptr;
            if (Inverse && pair && out && repair) {
                xy_repair<T>(src, full, *repair, out, s);
                screened = true;
                return;
            }
            if (pair && plane_pair<T, Inverse>(src, dst, full, act, axes[k], axes[k + 1], tune.pair_max,
                                               Inverse ? out : screen, s)) {
                ++k;
                screened = out != nullptr;
            } else {
                axis<T, Inverse>(src, dst, full, act, axes[k], tune.tile, screen, s);
            }
            src = dst;
        }
        if (src != final_dst) copy_box<T>(src, final_dst, full, act, s);
        first = false;
    }
};
}  // namespace

// ------------------------------------------------------------------ fused dyadic schedule
namespace {
// Leading levels whose box fills the GPU with fused workgroups (>= 512 of
// them at the smallest z segment); coarser boxes are cheaper as axis passes.
unsigned fused_levels(Dims n, unsigned levels) {
    unsigned f = 0;
    for (; f < levels; ++f) {
        const uint64_t wgs = uint64_t((n.nx + 63) / 64) * ((n.ny + 31) / 32) * ((n.nz + 15) / 16);
        if (wgs < 512) break;
        n = shrink(n, true, true);
    }
    return f;
}

// ------------------------------------------------------------------ tuning
// Launch choices of the dyadic schedule that do not change a single bit: how
// many leading levels run as fused kernels and each fused level's z segment.
// Per (geometry, type, direction): measured by autotune(), set explicitly, or
// the heuristic above.
struct TuneKey {
    uint32_t nx, ny, nz, width, inverse;
    bool operator<(const TuneKey& o) const {
        return std::tie(nx, ny, nz, width, inverse) < std::tie(o.nx, o.ny, o.nz, o.width, o.inverse);
    }
};
std::mutex g_tune_mu;
std::map<TuneKey, Tuning> g_tune;

// Workgroups of a fused level that share a CU (LDS: 42 KiB forward, 44-61 KiB
// inverse in float, twice that in double); constants, so that the choice needs
// no device.
Tuning heuristic_impl(Dims full, unsigned lxy, unsigned width, bool inverse) {
    constexpr uint32_t kCus = 256;
    const uint32_t per_cu = width == 8 ? 1 : inverse ? 2 : 3;
    Tuning t{};
    t.fused = fused_levels(full, lxy);
    t.tile[0] = t.tile[1] = t.tile[2] = 8;
    t.pair_max = 1024;
    Dims n = full;
    for (unsigned l = 0; l < 5; ++l) {
        t.sz[l] = best_z_segment(n, kCus, per_cu, 8);
        n = shrink(n, true, true);
    }
    return t;
}
// Compact boxes of levels >= 1 live in `scratch`: level l's box at offset 0
// for odd l and after the largest level-1 box for even l (two never-aliasing
// halves, each <= n/8 + lines).
template <class T>
T* low_box(T* scratch, Dims full, unsigned l) {
    const Dims h{half_len(full.nx), half_len(full.ny), half_len(full.nz)};
    const uint64_t first = uint64_t(h.nx) * h.ny * h.nz;
    return (l & 1u) ? scratch : scratch + ((first + 63) & ~uint64_t(63));
}
}  // namespace

Tuning tuning_for(Dims full, unsigned lxy, unsigned width, bool inverse) {
    std::lock_guard<std::mutex> g(g_tune_mu);
    const auto it = g_tune.find(TuneKey{full.nx, full.ny, full.nz, width, inverse ? 1u : 0u});
    Tuning t = it != g_tune.end() ? it->second : heuristic_impl(full, lxy, width, inverse);
    if (t.fused > lxy) t.fused = lxy;
    if (!fused_plane_fits(full.nx, full.ny, width)) t.fused = 0;  // planes of 4 GiB and more: axis passes
    return t;
}

Tuning heuristic_tuning(Dims full, unsigned lxy, unsigned width, bool inverse) {
    return heuristic_impl(full, lxy, width, inverse);
}

void clear_tuning() {
    std::lock_guard<std::mutex> g(g_tune_mu);
    g_tune.clear();
}

void set_tuning(Dims full, unsigned width, bool inverse, const Tuning& t) {
    for (unsigned l = 0; l < 5; ++l)
        if (t.sz[l] < 16 || t.sz[l] % 16) throw std::invalid_argument("z segment must be a positive multiple of 16");
    if (t.fused > 5) throw std::invalid_argument("at most five fused levels");
    for (unsigned a = 0; a < 3; ++a)
        if (t.tile[a] != 8 && t.tile[a] != 16 && t.tile[a] != 32)
            throw std::invalid_argument("pass tile must be 8, 16 or 32");
    if (t.pair_max != 0 && t.pair_max != 1024 && t.pair_max != 4096)
        throw std::invalid_argument("LDS pair limit must be 0, 1024 or 4096");
    std::lock_guard<std::mutex> g(g_tune_mu);
    g_tune[TuneKey{full.nx, full.ny, full.nz, width, inverse ? 1u : 0u}] = t;
}

std::string tuning_report() {
    std::lock_guard<std::mutex> g(g_tune_mu);
    std::string out = "[";
    for (const auto& [k, t] : g_tune) {
        if (out.size() > 1) out += ",";
        out += "{\"shape_xyz\":[" + std::to_string(k.nx) + "," + std::to_string(k.ny) + "," + std::to_string(k.nz) +
               "],\"width\":" + std::to_string(k.width) + ",\"inverse\":" + (k.inverse ? "true" : "false") +
               ",\"fused_levels\":" + std::to_string(t.fused) + ",\"z_segment\":[";
        for (unsigned l = 0; l < 5; ++l) out += (l ? "," : "") + std::to_string(t.sz[l]);
        out += "],\"pass_tiles_xyz\":[" + std::to_string(t.tile[0]) + "," + std::to_string(t.tile[1]) + "," +
               std::to_string(t.tile[2]) + "],\"lds_pair_max\":" + std::to_string(t.pair_max) + "}";
    }
    return out + "]";
}

template <class T>
void fused_forward(const T* input, T* coeff, T* tmp0, Dims full, unsigned levels, const Tuning& tu, uint32_t* status,
                   hipStream_t s) {
    const T* src = input;
    uint64_t spy = full.nx, spz = uint64_t(full.nx) * full.ny;
    Dims n = full;
    static const char* names[] = {"forward_L0", "forward_L1", "forward_L2", "forward_L3", "forward_L4"};
    for (unsigned l = 0; l < levels; ++l) {
        StageClock clock(names[l], s);
        const Dims h{half_len(n.nx), half_len(n.ny), half_len(n.nz)};
        FwdLevel<T> a;
        a.src = src;
        a.spy = spy;
        a.spz = spz;
        a.n = n;
        a.hi = coeff;
        a.hpy = full.nx;
        a.hpz = uint64_t(full.nx) * full.ny;
        if (l + 1 == levels) {
            a.lo = coeff;
            a.lpy = a.hpy;
            a.lpz = a.hpz;
        } else {
            a.lo = low_box(tmp0, full, l + 1);
            a.lpy = h.nx;
            a.lpz = uint64_t(h.nx) * h.ny;
        }
        a.sz = tu.sz[l];
        a.status = l == 0 ? status : nullptr;
        launch_fwd_level<T>(a, s);
        src = a.lo;
        spy = a.lpy;
        spz = a.lpz;
        n = h;
    }
}

// The finest inverse level as a fused kernel: high bands from `coeff`, the
// coarser reconstruction from `lo` (pitches lpy, lpz), into `output`, with
// the caller's emitter (store, screen and folded repairs, or the repair
// emitter, which may requantize the high bands on load).
template <class T>
void launch_finest(const T* coeff, const T* lo, uint32_t lpy, uint32_t lpz, T* output, Dims full, uint32_t sz,
                   const Level0Emit<T>* emit, hipStream_t s, const char* name) {
    const bool repairs = emit && emit->mode == kEmitRepair;
    const bool patch = emit && emit->mode == kEmitStoreScreen && emit->np;
    const uint64_t keys = patch ? patch_table_words(full, emit->np, sizeof(T)) : 0;
    if (!keys && patch) throw std::logic_error("repair list cannot be folded into the finest level");
    if (patch && !emit->ptable_built && emit->plan) throw std::logic_error("planned repair keys not built");
    if (patch && !emit->ptable_built) {  // the key table of the repairs the finest level applies
        StageClock clock("patch_keys", s);
        repair_keys<T>(emit->pidx, emit->perr, emit->np, full, emit->ptable, emit->status, s);
    }
    StageClock clock(repairs ? "inverse_L0_repairs" : name, s);
    InvLevel<T> a{};
    a.hi = coeff;
    a.hpy = full.nx;
    a.hpz = uint64_t(full.nx) * full.ny;
    a.lo = lo;
    a.lpy = lpy;
    a.lpz = lpz;
    a.n = full;
    a.out = output;
    a.opy = full.nx;
    a.opz = uint64_t(full.nx) * full.ny;
    a.sz = sz;
    a.emit = kEmitStore;
    if (emit) {
        a.emit = emit->mode;
        a.status = emit->status;
        a.orig = emit->orig;
        a.bound = emit->bound;
        if (repairs && emit->quantum > 0) {
            a.q = T(emit->quantum);
            a.inv = T(1.0 / emit->quantum);
        }
        a.bound_lo = float(emit->bound);
        if (double(a.bound_lo) > emit->bound) a.bound_lo = std::nextafter(a.bound_lo, 0.0f);
        a.rep = emit->rep;
        if (patch) {
            a.pidx = emit->pidx;
            a.perr = emit->perr;
            a.ptable = emit->ptable;
            a.np = emit->np;
            a.keys = uint32_t(keys);
            a.plan = emit->plan;
            a.archive = emit->archive;
        }
        if (repairs) {  // the segment layout the caller allocated fixes the z segment
            a.sz = emit->rep.cap / (64u * 32u);
            if (a.sz % 16 || inv_segments(full, a.sz) != emit->rep.segments)
                throw std::logic_error("repair segments do not match the finest level's launch");
        }
    }
    launch_inv_level<T>(a, s);
}

// Fused levels levels-1 .. 1 (the coarse LLL read from coeff): where their
// reconstruction of the level-1 box lies (coeff itself when only the finest
// level is fused).
template <class T>
LowBox<T> fused_coarse(T* coeff, T* tmp0, Dims full, unsigned levels, const Tuning& tu, hipStream_t s,
                       unsigned base) {
    Dims sizes[5], n = full;
    for (unsigned l = 0; l < levels; ++l) { sizes[l] = n; n = shrink(n, true, true); }
    LowBox<T> low{coeff, full.nx, full.nx * full.ny};
    static const char* names[] = {"inverse_L0", "inverse_L1", "inverse_L2", "inverse_L3", "inverse_L4"};
    for (int l = int(levels) - 1; l >= 1; --l) {
        StageClock clock(names[l + base], s);
        InvLevel<T> a{};
        a.hi = coeff;
        a.hpy = full.nx;
        a.hpz = uint64_t(full.nx) * full.ny;
        a.lo = low.p;
        a.lpy = low.py;
        a.lpz = low.pz;
        a.n = sizes[l];
        a.out = low_box(tmp0, full, unsigned(l));
        a.opy = sizes[l].nx;
        a.opz = uint64_t(sizes[l].nx) * sizes[l].ny;
        a.sz = tu.sz[l];
        a.emit = kEmitStore;
        launch_inv_level<T>(a, s);
        low = LowBox<T>{a.out, a.opy, a.opz};
    }
    return low;
}

template <class T>
void fused_inverse(T* coeff, T* output, T* tmp0, Dims full, unsigned levels, const Tuning& tu,
                   const Level0Emit<T>* emit, hipStream_t s, unsigned base) {
    static const char* names[] = {"inverse_L0", "inverse_L1", "inverse_L2", "inverse_L3", "inverse_L4"};
    const LowBox<T> low = fused_coarse<T>(coeff, tmp0, full, levels, tu, s, base);
    launch_finest<T>(coeff, low.p, low.py, low.pz, output, full, tu.sz[0], emit, s, names[base]);
}

RepairSegments level0_repair_segments(Dims full, unsigned lxy, unsigned lz, bool dyadic, unsigned width) {
    if (!dyadic && plane_fused_fits(full, lxy, lz, width))  // the Z phase detects them, by rows of columns
        return {full.ny * ((full.nx + kZColumns - 1) / kZColumns), std::min(full.nx, kZColumns) * full.nz,
                (full.nx & 31u) != 0};
    if (!dyadic || !lxy) return {};
    const Tuning tu = tuning_for(full, lxy, width, true);
    if (tu.fused) {
        const uint32_t sz =
            width == 4 ? repair_z_segment<float>(full, tu.sz[0]) : repair_z_segment<double>(full, tu.sz[0]);
        return {uint32_t(inv_segments(full, sz)), 64u * 32u * sz, (full.nx & 31u) != 0};
    }
    if (!strips_fit(full, full.nx, full.ny, 1, width)) return {};
    const StripPlan p = width == 4 ? repair_plan<float>(full) : repair_plan<double>(full);
    return {uint32_t(p.items()), strip_repair_cap(p), true};
}

// Full multi-level transform (cpu/src/transform.cpp:409-456).
// Forward: reads `input` (may equal coeff), leaves coefficients in `coeff`.
// Inverse: reads coefficients in `coeff` (overwritten), writes the last pass
// into `output` (may equal coeff). tmp0/tmp1: two full-volume scratch arrays.
template <class T>
void transform_forward(const T* input, T* coeff, T* tmp0, T* tmp1, Dims full, unsigned lxy, unsigned lz,
                       bool dyadic, uint32_t* status, hipStream_t s) {
    Passes<T, false> p{coeff, {tmp0, tmp1}, input, nullptr, status, s, tuning_for(full, lxy, sizeof(T), false)};
    if (lxy == 0 && lz == 0) {
        if (input != coeff) copy_box<T>(input, coeff, full, full, s);
        return;
    }
    if (dyadic) {
        const Tuning tu = tuning_for(full, lxy, sizeof(T), false);
        const unsigned fused = tu.fused;
        Dims act = full;
        if (fused) {
            if (input == coeff) {  // the level-0 kernel must not read what it writes
                copy_box<T>(input, tmp1, full, full, s);
                input = tmp1;
            }
            fused_forward<T>(input, coeff, tmp0, full, fused, tu, status, s);  // leaves LLL in coeff
            p.first = false;
            for (unsigned l = 0; l < fused; ++l) act = shrink(act, true, true);
        }
        static const int yxz[3] = {1, 0, 2};
        const unsigned tail = tail_level(full, lxy, fused, sizeof(T));
        for (unsigned l = fused; l < tail; ++l) {
            p.level(full, act, yxz, 3, false, l);
            act = shrink(act, true, true);
        }
        if (tail < lxy) {
            Tail<T> t = make_tail<T>(coeff, tmp0, full, tail, lxy);
            if (p.first) {  // the whole field: reads the input
                t.first = input;
                t.status = status;
            }
            tail_forward<T>(t, s);
        }
        return;
    }
    static const int zonly[1] = {2};
    static const int yx[2] = {1, 0};
    // every XY level as one launch of strips: the Z phase (one pass)
    // into tmp1, then level l reads its box (tmp1, then the compact boxes in
    // tmp0) and writes its high bands into coeff and its low band into the
    // next box (coeff for the last level)
    if (strip_lines_fit(full, lxy) && fused_plane_fits(full.nx, 1, sizeof(T)) && lxy &&
        (lz ? zcol_fits(full, lz, sizeof(T)) : input != coeff)) {
        const T* src = input;
        uint64_t spy = full.nx, spz = uint64_t(full.nx) * full.ny;
        if (lz) {
            StageClock clock("forward_Z", s);
            zcol_levels<T, false>(input, tmp1, full, lz, status, s);
            src = tmp1;
        }
        Dims n = full;
        static const char* names[] = {"forward_L0", "forward_L1", "forward_L2", "forward_L3", "forward_L4"};
        const unsigned tail = plane_tail_level(full, lxy);
        PlaneTail<T, XYForward<T>> pt{};
        for (unsigned l = 0; l < lxy; ++l) {
            StageClock clock(names[l], s);
            const Dims h{half_len(n.nx), half_len(n.ny), n.nz};
            const bool last = l + 1 == lxy;
            XYForward<T> a{src, spy, spz, coeff, full.nx, uint64_t(full.nx) * full.ny, nullptr, 0, 0, n,
                           l == 0 && !lz ? status : nullptr};
            a.lo = last ? coeff : xy_box(tmp0, full, l + 1);
            a.lpy = last ? full.nx : h.nx;
            a.lpz = last ? uint64_t(full.nx) * full.ny : uint64_t(h.nx) * h.ny;
            if (l < tail) xy_forward<T>(a, s);
            else add_plane(pt, a);
            src = a.lo;
            spy = a.lpy;
            spz = a.lpz;
            n = h;
        }
        if (pt.levels) {
            StageClock clock("forward_tail", s);
            hipLaunchKernelGGL((plane_tail_forward_kernel<T, false>), dim3(full.nz), dim3(64 * kPlaneTailWaves), 0, s, pt);
        }
        return;
    }
    Dims act = full;
    if (lz && zcol_fits(full, lz, sizeof(T))) {  // the Z phase in one pass
        StageClock clock("forward_Z", s);
        const T* src = z_source<T>(p.first_src, coeff, tmp0, full, lz, s);
        zcol_levels<T, false>(src, coeff, full, lz, status, s);
        p.first = false;
    } else {
        for (unsigned l = 0; l < lz; ++l) {
            p.level(full, act, zonly, 1, false, l);
            act = shrink(act, false, true);
        }
    }
    act = full;
    for (unsigned l = 0; l < lxy; ++l) {
        p.level(full, act, yx, 2, false, l);
        act = shrink(act, true, false);
    }
}

namespace {
template <class T>
WaveRepair<T> wave_repair(const Level0Emit<T>& e) {
    T lo = T(e.bound);
    if (double(lo) > e.bound) lo = std::nextafter(lo, T(0));
    return WaveRepair<T>{e.orig, e.bound, lo, e.rep};
}

// The dyadic levels lxy - 1 .. fused: the tail, then as passes; level 0 (none
// fused) ends as `p` says (its destination, screen or repairs).
template <class T>
void coarse_passes(Passes<T, true>& p, Dims full, unsigned lxy, unsigned fused, const Dims* sizes) {
    static const int zxy[3] = {2, 0, 1};
    const unsigned tail = tail_level(full, lxy, fused, sizeof(T));
    if (tail < lxy) {
        Tail<T> t = make_tail<T>(p.home, p.tmp[0], full, tail, lxy);
        if (tail == 0) {
            if (p.last_dst) t.last = p.last_dst;
            t.status = p.out_status;
            p.screened = p.out_status != nullptr;
        }
        tail_inverse<T>(t, full, tail == 0 ? p.repair : nullptr, p.s);
        p.first = false;
    }
    for (int l = int(tail) - 1; l >= int(fused); --l) p.level(full, sizes[l], zxy, 3, !fused && l == 0, unsigned(l));
}

// The inverse with launch choices `tu`; `base`: the level number of this
// field's level 0 (a coarse box run as a field of its own), for stage names.
template <class T>
bool inverse_impl(T* coeff, T* output, T* tmp0, T* tmp1, Dims full, unsigned lxy, unsigned lz, bool dyadic,
                  hipStream_t s, const Level0Emit<T>* emit, const Tuning& tu, unsigned base, double requant = 0.0) {
    if (requant > 0 && (dyadic || !plane_fused_fits(full, lxy, lz, sizeof(T))))
        throw std::logic_error("requantizing inverse without XY strips");
    Passes<T, true> p{coeff, {tmp0, tmp1}, coeff, output == coeff ? nullptr : output, nullptr, s, tu};
    p.base = base;
    if (lxy == 0 && lz == 0) {
        if (output != coeff) copy_box<T>(coeff, output, full, full, s);
        return false;
    }
    if (dyadic) {
        const unsigned fused = tu.fused;
        Dims sizes[5], act = full;
        for (unsigned l = 0; l < lxy; ++l) { sizes[l] = act; act = shrink(act, true, true); }
        // coarse levels as passes in coeff; then the fused levels (coarse LLL read from coeff)
        WaveRepair<T> repair{};
        if (!fused && emit && emit->mode == kEmitStoreScreen && !emit->np) p.out_status = emit->status;
        if (!fused && emit && emit->mode == kEmitRepair) {
            p.out_status = emit->status;
            repair = wave_repair(*emit);
            p.repair = &repair;
        }
        coarse_passes(p, full, lxy, fused, sizes);
        if (!fused) return p.screened;
        if (output == coeff) {  // the level-0 kernel must not overwrite what it reads
            fused_inverse<T>(coeff, tmp1, tmp0, full, fused, tu, emit, s, base);
            if (!emit || emit->mode != kEmitRepair) copy_box<T>(tmp1, coeff, full, full, s);
        } else {
            fused_inverse<T>(coeff, output, tmp0, full, fused, tu, emit, s, base);
        }
        return emit != nullptr;
    }
    Dims xy[5], zs[5], act = full;
    for (unsigned l = 0; l < lxy; ++l) { xy[l] = act; act = shrink(act, true, false); }
    act = full;
    for (unsigned l = 0; l < lz; ++l) { zs[l] = act; act = shrink(act, false, true); }
    static const int xyo[2] = {0, 1};
    static const int zonly[1] = {2};
    // every XY level as one launch of strips: level l reads coeff's bands and the
    // coarser reconstruction (coeff's low quadrant for the coarsest level,
    // then the compact boxes in tmp0) and writes its box to tmp0, the finest
    // into tmp1, from which the Z phase (one pass) writes output
    if (strips_fit(full, full.nx, full.ny, lxy, sizeof(T)) && lxy &&
        (lz ? zcol_fits(full, lz, sizeof(T)) : output != coeff)) {
        // the Z phase screens the output when asked (no repairs to fold here)
        uint32_t* screen = emit && emit->mode == kEmitStoreScreen && !emit->np && lz ? emit->status : nullptr;
        const bool repair = emit && emit->mode == kEmitRepair && lz;
        static const char* names[] = {"inverse_L0", "inverse_L1", "inverse_L2", "inverse_L3", "inverse_L4"};
        const T* lo = coeff;
        uint64_t lpy = full.nx, lpz = uint64_t(full.nx) * full.ny;
        const int tail = int(plane_tail_level(full, lxy));
        PlaneTail<T, XYInverse<T>> pt{};
        for (int l = int(lxy) - 1; l >= 0; --l) {
            StageClock clock(names[l + base], s);
            XYInverse<T> a{coeff, full.nx, uint64_t(full.nx) * full.ny, lo, lpy, lpz, nullptr, 0, 0, xy[l],
                           T(requant), requant > 0 ? T(1.0 / requant) : T(0), uint32_t(lo == coeff)};
            if (l == 0) {
                a.out = lz ? tmp1 : output;
                a.opy = full.nx;
                a.opz = uint64_t(full.nx) * full.ny;
            } else {
                a.out = xy_box(tmp0, full, unsigned(l));
                a.opy = xy[l].nx;
                a.opz = uint64_t(xy[l].nx) * xy[l].ny;
            }
            if (l >= tail) {
                add_plane(pt, a);
                if (l == tail) {
                    const dim3 grid(full.nz), block(64 * kPlaneTailWaves);
                    if (requant > 0)
                        hipLaunchKernelGGL((plane_tail_inverse_kernel<T, true, false>), grid, block, 0, s, pt);
                    else
                        hipLaunchKernelGGL((plane_tail_inverse_kernel<T, false, false>), grid, block, 0, s, pt);
                }
            } else {
                xy_inverse<T>(a, s);
            }
            lo = a.out;
            lpy = a.opy;
            lpz = a.opz;
        }
        if (lz) {
            StageClock clock("inverse_Z", s);
            if (repair) {
                const WaveRepair<T> z = wave_repair(*emit);
                zcol_levels<T, true>(tmp1, output, full, lz, emit->status, s, &z);
            } else {
                zcol_levels<T, true>(tmp1, output, full, lz, screen, s);
            }
        }
        return screen != nullptr || repair;
    }
    for (int l = int(lxy) - 1; l >= 0; --l) p.level(full, xy[l], xyo, 2, lz == 0 && l == 0, unsigned(l));
    if (lz && zcol_fits(full, lz, sizeof(T))) {  // the Z phase in one pass
        StageClock clock("inverse_Z", s);
        const T* src = z_source<T>(p.first ? p.first_src : p.home, output, tmp0, full, lz, s);
        zcol_levels<T, true>(src, output, full, lz, nullptr, s);
    } else {
        for (int l = int(lz) - 1; l >= 0; --l) p.level(full, zs[l], zonly, 1, l == 0, unsigned(l));
    }
    return false;
}

uint64_t pad64(uint64_t v) { return (v + 63) & ~uint64_t(63); }
uint64_t volume(Dims d) { return uint64_t(d.nx) * d.ny * d.nz; }
}  // namespace

template <class T>
bool transform_inverse(T* coeff, T* output, T* tmp0, T* tmp1, Dims full, unsigned lxy, unsigned lz, bool dyadic,
                       hipStream_t s, const Level0Emit<T>* emit, double requant) {
    return inverse_impl<T>(coeff, output, tmp0, tmp1, full, lxy, lz, dyadic, s, emit,
                           tuning_for(full, lxy, sizeof(T), true), 0, requant);
}

template <class T>
LowBox<T> inverse_coarse_levels(T* coeff, T* tmp0, T* tmp1, Dims full, unsigned lxy, hipStream_t s) {
    const Tuning tu = tuning_for(full, lxy, sizeof(T), true);
    if (!lxy || !tu.fused) throw std::logic_error("inverse split without a fused finest level");
    Passes<T, true> p{coeff, {tmp0, tmp1}, coeff, nullptr, nullptr, s, tu};
    Dims sizes[5], act = full;
    for (unsigned l = 0; l < lxy; ++l) { sizes[l] = act; act = shrink(act, true, true); }
    coarse_passes(p, full, lxy, tu.fused, sizes);
    return fused_coarse<T>(coeff, tmp0, full, tu.fused, tu, s, 0);
}

template <class T>
void inverse_finest_level(const T* coeff, const LowBox<T>& low, T* output, Dims full, unsigned lxy,
                          const Level0Emit<T>& emit, hipStream_t s) {
    if (output == coeff) throw std::logic_error("the finest level must not overwrite its coefficients");
    const Tuning tu = tuning_for(full, lxy, sizeof(T), true);
    launch_finest<T>(coeff, low.p, low.py, low.pz, output, full, tu.sz[0], &emit, s, "inverse_L0");
}

template <class T>
bool transform_inverse_preserving(const T* coeff, T* output, T* tmp0, T* tmp1, Dims full, unsigned lxy, unsigned lz,
                                  bool dyadic, hipStream_t s) {
    if (output == coeff) return false;
    if (!dyadic) {
        if (lxy || !lz || !zcol_fits(full, lz, sizeof(T))) return false;
        StageClock clock("inverse_Z", s);
        zcol_levels<T, true>(coeff, output, full, lz, nullptr, s);
        return true;
    }
    const Tuning tu = tuning_for(full, lxy, sizeof(T), true);
    if (!lxy || !tu.fused) return false;
    const Dims h1 = shrink(full, true, true);
    // the coarser levels work on a copy of their box, with the output as a
    // scratch volume: the finest level reads their result as it stores
    copy_box<T>(coeff, tmp1, full, h1, s);
    const LowBox<T> low = inverse_coarse_levels<T>(tmp1, tmp0, output, full, lxy, s);
    if (low.p == output) throw std::logic_error("coarse levels ended in the output");
    const Level0Emit<T> store{kEmitStore, nullptr, nullptr, 0.0, SegList{}, 0.0};
    inverse_finest_level<T>(coeff, low, output, full, lxy, store, s);
    return true;
}

bool plane_fused_fits(Dims full, unsigned lxy, unsigned lz, unsigned width) {
    return lxy && lz && zcol_fits(full, lz, width) && strips_fit(full, full.nx, full.ny, lxy, width);
}

bool coarse_split_fits(Dims full, unsigned lxy, unsigned width) {
    if (lxy < 2 || tuning_for(full, lxy, width, true).fused < 2) return false;
    const Dims h1 = shrink(full, true, true), h2 = shrink(h1, true, true);
    return 4 * pad64(volume(h2)) <= volume(full) && volume(h1) <= volume(full);
}

template <class T>
void inverse_coarse_requant(const T* coeff, T* t0, T* t1, Dims full, unsigned lxy, double quantum, hipStream_t s) {
    if (!coarse_split_fits(full, lxy, sizeof(T))) throw std::logic_error("coarse inverse split does not apply");
    const Tuning tu = tuning_for(full, lxy, sizeof(T), true);
    const Dims h1 = shrink(full, true, true), h2 = shrink(h1, true, true);
    const uint64_t v2 = pad64(volume(h2));
    T *c2 = t1, *o2 = t1 + v2, *w0 = t1 + 2 * v2, *w1 = t1 + 3 * v2;
    const T q = T(quantum), inv = T(1.0 / quantum);
    {
        StageClock clock("coarse_requant", s);
        const uint64_t total = volume(h2);
        check_launch_size(total);
        hipLaunchKernelGGL((box_requant<T>), dim3(uint32_t((total + 255) / 256)), dim3(256), 0, s, coeff, c2, full, h2,
                           uint32_t(total), q, inv);
    }
    const T* lo = c2;
    if (lxy > 2) {  // levels >= 2: the box as a field of its own, with this field's launch choices
        Tuning t2 = tu;
        t2.fused = tu.fused - 2;
        for (unsigned l = 0; l < 5; ++l) t2.sz[l] = l + 2 < 5 ? tu.sz[l + 2] : 16u;
        inverse_impl<T>(c2, o2, w0, w1, h2, lxy - 2, lxy - 2, true, s, nullptr, t2, 2);
        lo = o2;
    }
    StageClock clock("inverse_L1", s);
    InvLevel<T> a{};
    a.hi = coeff;
    a.hpy = full.nx;
    a.hpz = uint64_t(full.nx) * full.ny;
    a.lo = lo;
    a.lpy = h2.nx;
    a.lpz = uint64_t(h2.nx) * h2.ny;
    a.n = h1;
    a.out = t0;
    a.opy = h1.nx;
    a.opz = uint64_t(h1.nx) * h1.ny;
    a.sz = tu.sz[1];
    a.emit = kEmitStore;
    a.q = q;
    a.inv = inv;
    launch_inv_level<T>(a, s);
}

template <class T>
void inverse_finest_requant(const T* coeff, const T* t0, Dims full, unsigned lxy, const Level0Emit<T>& emit,
                            hipStream_t s) {
    const Tuning tu = tuning_for(full, lxy, sizeof(T), true);
    const Dims h1 = shrink(full, true, true);
    launch_finest<T>(coeff, t0, h1.nx, h1.nx * h1.ny, nullptr, full, tu.sz[0], &emit, s, "inverse_L0");
}

template bool transform_inverse_preserving<float>(const float*, float*, float*, float*, Dims, unsigned, unsigned, bool,
                                                  hipStream_t);
template bool transform_inverse_preserving<double>(const double*, double*, double*, double*, Dims, unsigned, unsigned,
                                                   bool, hipStream_t);
template LowBox<float> inverse_coarse_levels<float>(float*, float*, float*, Dims, unsigned, hipStream_t);
template LowBox<double> inverse_coarse_levels<double>(double*, double*, double*, Dims, unsigned, hipStream_t);
template void inverse_finest_level<float>(const float*, const LowBox<float>&, float*, Dims, unsigned,
                                          const Level0Emit<float>&, hipStream_t);
template void inverse_finest_level<double>(const double*, const LowBox<double>&, double*, Dims, unsigned,
                                           const Level0Emit<double>&, hipStream_t);
template void transform_forward<float>(const float*, float*, float*, float*, Dims, unsigned, unsigned, bool,
                                       uint32_t*, hipStream_t);
template void transform_forward<double>(const double*, double*, double*, double*, Dims, unsigned, unsigned, bool,
                                        uint32_t*, hipStream_t);
template bool transform_inverse<float>(float*, float*, float*, float*, Dims, unsigned, unsigned, bool, hipStream_t,
                                       const Level0Emit<float>*, double);
template bool transform_inverse<double>(double*, double*, double*, double*, Dims, unsigned, unsigned, bool,
                                        hipStream_t, const Level0Emit<double>*, double);
template void inverse_coarse_requant<float>(const float*, float*, float*, Dims, unsigned, double, hipStream_t);
template void inverse_coarse_requant<double>(const double*, double*, double*, Dims, unsigned, double, hipStream_t);
template void inverse_finest_requant<float>(const float*, const float*, Dims, unsigned, const Level0Emit<float>&,
                                            hipStream_t);
template void inverse_finest_requant<double>(const double*, const double*, Dims, unsigned, const Level0Emit<double>&,
                                             hipStream_t);

}  // namespace wz
