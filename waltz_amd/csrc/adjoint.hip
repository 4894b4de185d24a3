// Adjoints (transposes) of the multi-level CDF 9/7 transforms, for gradients:
// DWT^T maps a coefficient-space gradient to sample space, IDWT^T maps a
// sample-space gradient to coefficient space. No reference counterpart.
//
// One axis pass of the forward transform lifts every line of the active box:
// the line is extended by whole-sample symmetric reflection, the four lifting
// steps and the scaling run on the extended sequence, and the result is
// restricted to [0, n) and split (even samples first, odd after). The lifting
// steps keep the reflection symmetry, so the pass equals
// split . restrict . L . reflect with L the lifting of an unbounded line. Its
// transpose is reflect^T . L^T . restrict^T . split^T: interleave the split
// gradient, extend it by zeros, run the transposed steps in reverse order
// (each "x[k] += c (x[k-1] + x[k+1])" on one parity becomes the same update on
// the other parity), and fold every extended position back onto the sample it
// reflects to. The inverse pass is the mirror image (split input, natural
// output). The support of L^T is 4 samples wide on each side, so a line chunk
// of 64 outputs is computed from a zero-extended window with 16 samples of
// margin staged in LDS, one 8-sample tile per thread in registers (from the
// tile's 16-sample neighbourhood), with no barrier between the updates.
//
// The adjoint of a multi-level transform runs the transposed passes in the
// reverse order of the transform's schedule. Each level is one XY launch (the
// strips of the transforms, Adjoint) and one Z launch, each reading and
// writing its box once; low boxes move on in compact copies, so no level is
// copied back. Against a pass per axis through LDS (and, on small planes, one
// for X and Y with a halo of 2.4 times its outputs), IDWT^T / DWT^T:
// 256^3 float 199 -> 106 / 234 -> 124 us, double 439 -> 184 / 508 -> 206;
// 203x150x61 double 142 -> 60 / 159 -> 68. Memory bounds the finest level,
// launches the coarse ones. The passes per axis (adjoint_pass) are left for
// lines of one sample and planes past a 32-bit window.
#include <algorithm>

#include "common.hpp"
#include "fused.hpp"
#include "launch.hpp"
#include "lifting.hpp"
#include "planetail.hpp"

namespace wz {
namespace {

constexpr int kChunkOut = 64;                  // outputs per line chunk
constexpr int kMargin = 16;                    // window margin on each side
constexpr int kWin = kChunkOut + 2 * kMargin;  // 96 window samples

WZ_HD uint32_t split_index(uint32_t p, uint32_t n) { return (p >> 1) + ((p & 1u) ? half_len(n) : 0u); }

// Lines per workgroup: X lines are rows (window along x); Y and Z lines are
// 32 consecutive x, so every global access is a 128-byte (f32) row segment.
constexpr int kLines = 32;

// Transposed lifting of one 8-sample tile (window positions [i0, i0 + 8))
// from its 16-sample neighbourhood [i0 - 4, i0 + 12) in registers: the four
// updates, each "x[k] += c (x[k-1] + x[k+1])" on one parity, lose one pair of
// validity at the tile ends, so pairs 2..5 of the 8 loaded are final. Every
// value is the same sequence of operations as the same update run over the
// whole window.
// (`ws`, `os`: element strides of the neighbourhood and the result).
template <class T, bool OfInverse>
WZ_D void tile_transposed(const T* w, T* out, int ws = 1, int os = 1) {
    using C = Lift<T>;
    T e[8], o[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        e[j] = w[(2 * j) * ws];
        o[j] = w[(2 * j + 1) * ws];
    }
    if constexpr (OfInverse) {  // transposes of A', B', G', D' in that order
#pragma unroll
        for (int j = 1; j < 8; ++j) e[j] = fmadd(-C::a, o[j - 1] + o[j], e[j]);
#pragma unroll
        for (int j = 1; j < 7; ++j) o[j] = fmadd(-C::b, e[j] + e[j + 1], o[j]);
#pragma unroll
        for (int j = 2; j < 7; ++j) e[j] = fmadd(-C::g, o[j - 1] + o[j], e[j]);
#pragma unroll
        for (int j = 2; j < 6; ++j) o[j] = fmadd(-C::d, e[j] + e[j + 1], o[j]);
    } else {  // transposes of D, G, B, A in that order (after the scaling)
#pragma unroll
        for (int j = 0; j < 7; ++j) o[j] = fmadd(C::d, e[j] + e[j + 1], o[j]);
#pragma unroll
        for (int j = 1; j < 7; ++j) e[j] = fmadd(C::g, o[j - 1] + o[j], e[j]);
#pragma unroll
        for (int j = 1; j < 6; ++j) o[j] = fmadd(C::b, e[j] + e[j + 1], o[j]);
#pragma unroll
        for (int j = 2; j < 6; ++j) e[j] = fmadd(C::a, o[j - 1] + o[j], e[j]);
    }
#pragma unroll
    for (int j = 2; j < 6; ++j) {
        out[(2 * (j - 2)) * os] = e[j];
        out[(2 * (j - 2) + 1) * os] = o[j];
    }
}

// OfInverse: transpose of the inverse pass (natural -> split), else of the
// forward pass (split -> natural).
template <class T, bool OfInverse, int Axis>
__global__ void __launch_bounds__(256) adjoint_pass(const T* __restrict__ src, T* __restrict__ dst, Dims full,
                                                    Dims act, uint32_t chunks, uint32_t groups) {
    constexpr int L = kLines;
    __shared__ T v[L][kWin + 1];
    // transposed-lifting results at positions [c0 - 8, c0 + 72): the chunk
    // and the extended positions the fold reads
    constexpr int kRes = kChunkOut + 16;
    __shared__ T r[L][kRes + 1];
    __shared__ uint64_t lbase[L];
    using C = Lift<T>;
    const uint32_t n = Axis == 0 ? act.nx : Axis == 1 ? act.ny : act.nz;
    const uint32_t chunk = blockIdx.x % chunks, rest = blockIdx.x / chunks;
    const uint32_t group = rest % groups, outer = rest / groups;
    const uint32_t c0 = chunk * kChunkOut;
    const uint64_t plane = uint64_t(full.nx) * full.ny;
    const uint64_t stride = Axis == 0 ? 1u : Axis == 1 ? uint64_t(full.nx) : plane;

    // line l of this workgroup: base offset, or ~0 when out of the box
    auto line_base = [&](uint32_t l) -> uint64_t {
        if constexpr (Axis == 0) {
            const uint64_t li = uint64_t(group) * L + l;
            if (li >= uint64_t(act.ny) * act.nz) return ~uint64_t(0);
            const uint32_t y = uint32_t(li % act.ny), z = uint32_t(li / act.ny);
            return uint64_t(z) * plane + uint64_t(y) * full.nx;
        } else {
            const uint32_t x = group * L + l;
            if (x >= act.nx) return ~uint64_t(0);
            return Axis == 1 ? uint64_t(outer) * plane + x : uint64_t(outer) * full.nx + x;
        }
    };

    if (threadIdx.x < uint32_t(L)) lbase[threadIdx.x] = line_base(threadIdx.x);
    __syncthreads();

    // zero-extended window [c0 - margin, c0 + 64 + margin) of the interleaved line
    for (uint32_t w = threadIdx.x; w < uint32_t(L * kWin); w += 256) {
        const uint32_t l = Axis == 0 ? w / kWin : w % L, i = Axis == 0 ? w % kWin : w / L;
        const int32_t q = int32_t(c0) - kMargin + int32_t(i);
        const uint64_t base = lbase[l];
        T x = T(0);
        if (base != ~uint64_t(0) && q >= 0 && uint32_t(q) < n) {
            const uint32_t pos = OfInverse ? uint32_t(q) : split_index(uint32_t(q), n);
            x = src[base + uint64_t(pos) * stride];
        }
        if (!OfInverse) x = (i & 1u) ? x * (-C::ik) : x * C::k;  // scaling first
        v[l][i] = x;
    }
    __syncthreads();
    // the chunk's 8 tiles of every line, one per thread; the tile before it
    // (images -p, p = 1..4, at the line start) and the one after it (images
    // 2n - 2 - p at the line end) only where those exist
    static_assert(L * (kChunkOut / 8) == 256, "one chunk tile per thread");
    auto tile = [&](uint32_t l, int k) {  // window positions [kMargin + 8k, +8)
        tile_transposed<T, OfInverse>(&v[l][kMargin + 8 * k - 4], &r[l][8 + 8 * k]);
    };
    tile(threadIdx.x % L, int(threadIdx.x / L));
    if (c0 == 0 && threadIdx.x < uint32_t(L)) tile(threadIdx.x, -1);
    if (c0 + kChunkOut + 8 > n && threadIdx.x >= uint32_t(L) && threadIdx.x < uint32_t(2 * L))
        tile(threadIdx.x - L, kChunkOut / 8);
    __syncthreads();

    // fold the extended positions onto the samples they reflect to
    const int32_t lo = -4, hi = int32_t(n) + 4;  // support of the transposed lifting
    for (uint32_t w = threadIdx.x; w < uint32_t(L * kChunkOut); w += 256) {
        const uint32_t l = Axis == 0 ? w / kChunkOut : w % L, i = Axis == 0 ? w % kChunkOut : w / L;
        const uint32_t p = c0 + i;
        const uint64_t base = lbase[l];
        if (base == ~uint64_t(0) || p >= n) continue;
        auto u = [&](int32_t q) { return r[l][q - int32_t(c0) + 8]; };
        T s = u(int32_t(p));
        if (n >= 9) {  // at most two more images: -p and 2n-2-p
            if (p >= 1 && p <= 4) s += u(-int32_t(p));
            const int32_t m = 2 * int32_t(n) - 2 - int32_t(p);
            if (m != int32_t(p) && m < hi) s += u(m);
        } else {  // short line: the whole window is one chunk
            for (int32_t q = lo; q < hi; ++q)
                if (q != int32_t(p) && reflect_pos(q, n) == p) s += u(q);
        }
        if (OfInverse && n == 1) {  // its one sample is every even and every odd one
            T even = T(0), odd = T(0);
            for (int32_t q = lo; q < hi; ++q) {
                if (q & 1) odd += u(q);
                else even += u(q);
            }
            s = even * C::ik + odd * (-C::k);
        } else if (OfInverse) {
            s = (p & 1u) ? s * (-C::k) : s * C::ik;
        }
        dst[base + uint64_t(OfInverse ? split_index(p, n) : p) * stride] = s;
    }
}

Dims shrink_box(Dims d, bool xy, bool z) {
    if (xy) {
        d.nx = half_len(d.nx);
        d.ny = half_len(d.ny);
    }
    if (z) d.nz = half_len(d.nz);
    return d;
}

template <class T, bool OfInverse, int Axis>
void launch_adjoint(const T* src, T* dst, Dims full, Dims act, hipStream_t s) {
    constexpr int L = kLines;
    const uint32_t n = Axis == 0 ? act.nx : Axis == 1 ? act.ny : act.nz;
    if (!n || !act.nx || !act.ny || !act.nz) return;
    const uint32_t chunks = (n + kChunkOut - 1) / kChunkOut;
    const uint64_t groups =
        Axis == 0 ? (uint64_t(act.ny) * act.nz + L - 1) / L : (uint64_t(act.nx) + L - 1) / L;
    const uint64_t outer = Axis == 0 ? 1u : Axis == 1 ? act.nz : act.ny;
    const uint64_t blocks = uint64_t(chunks) * groups * outer;
    check_launch_size(blocks * 256);
    hipLaunchKernelGGL((adjoint_pass<T, OfInverse, Axis>), dim3(uint32_t(blocks)), dim3(256), 0, s, src, dst, full,
                       act, chunks, uint32_t(groups));
}

template <class T, bool OfInverse>
void adjoint_axis(const T* src, T* dst, Dims full, Dims act, int axis, hipStream_t s) {
    if (axis == 0) launch_adjoint<T, OfInverse, 0>(src, dst, full, act, s);
    else if (axis == 1) launch_adjoint<T, OfInverse, 1>(src, dst, full, act, s);
    else launch_adjoint<T, OfInverse, 2>(src, dst, full, act, s);
}

template <class T>
__global__ void __launch_bounds__(256) adjoint_copy(const T* __restrict__ src, T* __restrict__ dst, Dims full,
                                                    Dims act, uint32_t total) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= total) return;
    const uint32_t x = i % act.nx, r = i / act.nx, y = r % act.ny, z = r / act.ny;
    const uint64_t at = (uint64_t(z) * full.ny + y) * full.nx + x;
    dst[at] = src[at];
}

// ------------------------------------------------------------------ levels in registers
// OfInverse: the transpose of the inverse's level (natural -> split), else of
// the forward's (split -> natural).
template <class T, bool OfInverse>
__global__ void __launch_bounds__(kStripThreads) adjoint_xy_kernel(std::conditional_t<OfInverse, XYForward<T>,
                                                                                      XYInverse<T>> a, StripPlan p) {
    uint32_t item;
    if (!strip_of_wave(p, item)) return;
    if constexpr (OfInverse) strip_forward<T, true>(a, p, item);
    else strip_inverse<T, false, true>(a, p, item, StripStore<T>{});
}

// One Z level of a box. `nat`: its samples along z; `lo`: the low planes of
// the columns x < lx, y < ly; `hi`: everything else of the split.
template <class T>
struct ZLevel {
    T* nat;  // read by OfInverse, else written; the other two the other way round
    uint64_t npy, npz;
    T* hi;
    uint64_t hpy, hpz;
    T* lo;
    uint64_t lpy, lpz;
    Dims n;
    uint32_t lx, ly;
    uint32_t sz, groups, items;  // planes of a segment, waves per segment, waves
};

// A lane streams one column of the box (columns counted row by row), two
// planes a step, as the strips stream rows; ends as there (mirror_lift).
template <class T, bool OfInverse>
__global__ void __launch_bounds__(256) adjoint_z_kernel(ZLevel<T> a) {
    using C = Lift<T>;
    constexpr uint32_t S = sizeof(T);
    const uint32_t per = ((a.items + 3) / 4 + 7) / 8;
    const uint32_t item = 4 * ((blockIdx.x & 7u) * per + (blockIdx.x >> 3)) +
                          __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (item >= a.items || (blockIdx.x >> 3) >= per) return;
    const uint32_t seg = item / a.groups, c = (item - seg * a.groups) * 64u + (threadIdx.x & 63u);
    const Dims n = a.n;
    const int32_t nz = int32_t(n.nz);
    const uint32_t hz = half_len(n.nz);
    const bool live = c < n.nx * n.ny;
    const uint32_t y = live ? c / n.nx : 0u, x = live ? c - y * n.nx : 0u;
    const bool low = x < a.lx && y < a.ly;
    // one plane's windows; lanes outside go past their range (loads 0, stores
    // dropped)
    const uint32_t nr = ((n.ny - 1u) * uint32_t(a.npy) + n.nx) * S, hr = ((n.ny - 1u) * uint32_t(a.hpy) + n.nx) * S;
    const uint32_t lr = ((a.ly - 1u) * uint32_t(a.lpy) + a.lx) * S;
    auto natural = [&](T* p, uint32_t z) { return window_n(p + uint64_t(z) * a.npz, nr); };
    auto high = [&](T* p, uint32_t z) { return window_n(p + uint64_t(z) * a.hpz, hr); };
    auto lower = [&](T* p, uint32_t z) { return window_n(p + uint64_t(z) * a.lpz, lr); };
    const uint32_t nv = live ? (y * uint32_t(a.npy) + x) * S : kOutside;
    const uint32_t hv = live ? (y * uint32_t(a.hpy) + x) * S : kOutside;
    const uint32_t lv = live && low ? (y * uint32_t(a.lpy) + x) * S : kOutside;
    const uint32_t hl = low ? kOutside : hv;  // this column's low planes in `hi`
    const bool some = __ballot(live && !low) != 0;
    const uint32_t zs = seg * a.sz, blocks = (min(a.sz, n.nz - zs) + 7) / 8;
    auto load = [&](int32_t g, T (&v)[2]) {
        const uint32_t pe = uint32_t(pair_even(g, nz)), po = uint32_t(pair_odd(g, nz));
        if constexpr (OfInverse) {
            v[0] = buf_load<T>(natural(a.nat, 2 * pe), nv);
            v[1] = buf_load<T>(natural(a.nat, 2 * po + 1), nv);
        } else {
            v[0] = buf_load<T>(lower(a.lo, pe), lv);
            if (some) {
                const T h = buf_load<T>(high(a.hi, pe), hl);
                v[0] = low ? v[0] : h;
            }
            v[1] = buf_load<T>(high(a.hi, hz + po), hv);
        }
    };
    T s0 = T(0), s1 = T(0), s2 = T(0), s3 = T(0), s4 = T(0);  // the pipeline's states
    T buf[4][2];
    int32_t g = int32_t(zs / 2) - 2;
    load(g, buf[0]);
    load(g + 1, buf[1]);
    load(g + 2, buf[2]);
    const uint32_t images = line_images(nz);
    auto block = [&](bool emit) {
#pragma unroll
        for (int u = 0; u < 4; ++u, ++g) {
            load(g + 3, buf[(u + 3) & 3]);
            const uint32_t k = uint32_t(g - 2);
            const T e = buf[u][0], o = buf[u][1];
            T r0, r1;  // pair g - 2
            mirror_stream(g, nz, images, [&](const MirrorSteps& m, auto ends_c) {
                constexpr bool ends = decltype(ends_c)::value;
                if constexpr (OfInverse) {
                    const T e1 = mirror_lift<ends>(-C::a, s0, o, e, m, 5);
                    const T o1 = mirror_lift<ends>(-C::b, s1, e1, s0, m, 4);
                    const T e2 = mirror_lift<ends>(-C::g, s2, o1, s1, m, 3);
                    r0 = s3 * C::ik;
                    r1 = mirror_lift<ends>(-C::d, s3, e2, s2, m, 2) * (-C::k);
                    s0 = o;
                    s1 = e1;
                    s2 = o1;
                    s3 = e2;
                } else {
                    const T ev = e * C::k, ov = o * (-C::ik);
                    const T o1 = mirror_lift<ends>(C::d, s4, ev, s0, m, 4);
                    const T e1 = mirror_lift<ends>(C::g, s1, o1, s4, m, 3);
                    const T o2 = mirror_lift<ends>(C::b, s2, e1, s1, m, 2);
                    r0 = mirror_lift<ends>(C::a, s3, o2, s2, m, 1);
                    r1 = o2;
                    s4 = ev;
                    s0 = ov;
                    s1 = o1;
                    s2 = e1;
                    s3 = o2;
                }
            });
            if (!emit) continue;
            if constexpr (OfInverse) {
                if (2 * k < n.nz) {
                    buf_store(r0, lower(a.lo, k), lv);
                    if (some) buf_store(r0, high(a.hi, k), hl);
                }
                if (2 * k + 1 < n.nz) buf_store(r1, high(a.hi, hz + k), hv);
            } else {
                if (2 * k < n.nz) buf_store(r0, natural(a.nat, 2 * k), nv);
                if (2 * k + 1 < n.nz) buf_store(r1, natural(a.nat, 2 * k + 1), nv);
            }
        }
    };
    block(false);
    for (uint32_t b = 0; b < blocks; ++b) block(true);
}

// A box and where it lies.
template <class T>
struct Box {
    T* p;
    uint64_t py, pz;
};
template <class T>
Box<T> volume(T* p, Dims full) { return {p, full.nx, uint64_t(full.nx) * full.ny}; }
template <class T>
Box<T> compact(T* p, Dims n) { return {p, n.nx, uint64_t(n.nx) * n.ny}; }

// in: the samples' gradient (OfInverse) or the split one, its low box `lo`
template <class T, bool OfInverse>
using XYLevel = std::conditional_t<OfInverse, XYForward<T>, XYInverse<T>>;
template <class T, bool OfInverse>
XYLevel<T, OfInverse> level_of(Box<T> in, Box<T> lo, Box<T> out, Dims n) {
    if constexpr (OfInverse) return {in.p, in.py, in.pz, out.p, out.py, out.pz, lo.p, lo.py, lo.pz, n, nullptr};
    else return {in.p, in.py, in.pz, lo.p, lo.py, lo.pz, out.p, out.py, out.pz, n, T(0), T(0), 0u};
}
template <class T, bool OfInverse>
void xy_level(Box<T> in, Box<T> lo, Box<T> out, Dims n, hipStream_t s) {
    const StripPlan p = strip_plan(n, strips_pack(std::max({in.pz, lo.pz, out.pz}), sizeof(T)));
    hipLaunchKernelGGL((adjoint_xy_kernel<T, OfInverse>), dim3(strip_blocks(p)), dim3(kStripThreads), 0, s,
                       (level_of<T, OfInverse>(in, lo, out, n)), p);
}
template <class T, bool OfInverse>
void xy_tail(const PlaneTail<T, XYLevel<T, OfInverse>>& t, uint32_t planes, hipStream_t s) {
    const dim3 grid(planes), block(64 * kPlaneTailWaves);
    if constexpr (OfInverse) hipLaunchKernelGGL((plane_tail_forward_kernel<T, true>), grid, block, 0, s, t);
    else hipLaunchKernelGGL((plane_tail_inverse_kernel<T, false, true>), grid, block, 0, s, t);
}
// nat: the samples along z; hi, lo: the split and its low box of lx x ly columns
template <class T, bool OfInverse>
void z_level(Box<T> nat, Box<T> hi, Box<T> lo, Dims n, uint32_t lx, uint32_t ly, hipStream_t s) {
    ZLevel<T> a{nat.p, nat.py, nat.pz, hi.p, hi.py, hi.pz, lo.p, lo.py, lo.pz, n, lx, ly, 128, 0, 0};
    a.groups = uint32_t((uint64_t(n.nx) * n.ny + 63) / 64);
    auto waves = [&] { return uint64_t(a.groups) * ((n.nz + a.sz - 1) / a.sz); };
    while (a.sz > 32 && waves() < 8192) a.sz >>= 1;
    if (waves() < 1024) a.sz = 16;
    const uint64_t blocks = 8 * (((waves() + 3) / 4 + 7) / 8);
    check_launch_size(blocks * 256);
    a.items = uint32_t(waves());
    hipLaunchKernelGGL((adjoint_z_kernel<T, OfInverse>), dim3(uint32_t(blocks)), dim3(256), 0, s, a);
}

// Whether every level runs in registers: no line of one sample, planes inside
// one 32-bit window.
bool levels_fit(Dims full, unsigned lxy, unsigned lz, unsigned width) {
    uint32_t z = full.nz;
    for (unsigned l = 0; l < lz; ++l, z = half_len(z))
        if (z < 2) return false;
    return full.nx && full.ny && full.nz && strips_fit(full, full.nx, full.ny, lxy, width);
}

// The transforms' schedules reversed, from `src` into `data` (which may be the
// same). The high bands of a level go to (or come from) their place in a full
// volume, its low box to a compact one in tmp1: odd levels' at its start, even
// ones' after the largest odd one (lines of at least 2 samples: both fit), the
// plane schedule's XY boxes one after the other.
template <class T, bool OfInverse>
void adjoint_levels(T* data, const T* src, T* tmp0, T* tmp1, Dims full, unsigned lxy, unsigned lz, bool dyadic,
                    hipStream_t s) {
    T* from = const_cast<T*>(src);  // (only read unless it is data)
    auto low_of = [&](unsigned l, bool xy, bool z) {  // the compact box of level l >= 1
        const Dims h = shrink_box(full, xy, z);
        Dims n = full;
        for (unsigned k = 0; k < l; ++k) n = shrink_box(n, xy, z);
        return compact(tmp1 + ((l & 1u) ? 0u : uint64_t(h.nx) * h.ny * h.nz), n);
    };
    auto box_of = [&](unsigned l, bool xy, bool z) {
        Dims n = full;
        for (unsigned k = 0; k < l; ++k) n = shrink_box(n, xy, z);
        return n;
    };
    const Box<T> home = volume(data, full);
    if (dyadic) {
        for (unsigned k = 0; k < lxy; ++k) {
            const unsigned l = OfInverse ? k : lxy - 1 - k;
            const Dims n = box_of(l, true, true);
            const uint32_t lx = half_len(n.nx), ly = half_len(n.ny);
            const bool last = l + 1 == lxy;
            const Box<T> mid = compact(tmp0, n);
            if constexpr (OfInverse) {
                const Box<T> in = l ? low_of(l, true, true) : volume(from, full);
                xy_level<T, true>(in, mid, mid, n, s);
                z_level<T, true>(mid, home, last ? home : low_of(l + 1, true, true), n, lx, ly, s);
            } else {
                const Box<T> hi = volume(from, full);
                z_level<T, false>(mid, hi, last ? hi : low_of(l + 1, true, true), n, lx, ly, s);
                xy_level<T, false>(mid, mid, l ? low_of(l, true, true) : home, n, s);
            }
        }
        return;
    }
    // one of the two phases only: it must not write the volume it reads
    if (from == data && (!lxy || !lz)) {
        hip_check(hipMemcpyAsync(tmp0, data, uint64_t(full.nx) * full.ny * full.nz * sizeof(T),
                                 hipMemcpyDeviceToDevice, s),
                  "copy");
        from = tmp0;
    }
    const Box<T> mid = lxy && lz ? volume(tmp0, full) : home;  // between the two phases
    auto z_phase = [&](Box<T> in, Box<T> out) {
        for (unsigned k = 0; k < lz; ++k) {
            const unsigned l = OfInverse ? k : lz - 1 - k;
            const Dims n = box_of(l, false, true);
            const bool last = l + 1 == lz;
            const Box<T> split = OfInverse ? out : in;
            const Box<T> nat = l ? low_of(l, false, true) : OfInverse ? in : out;
            z_level<T, OfInverse>(nat, split, last ? split : low_of(l + 1, false, true), n, n.nx, n.ny, s);
        }
    };
    // (the tail takes each plane through several levels: no two levels' boxes
    // may share memory)
    auto plane_box = [&](unsigned l) { return compact(xy_box(tmp1, full, l), box_of(l, true, false)); };
    auto xy_phase = [&](Box<T> in, Box<T> out) {
        const unsigned tail = plane_tail_level(full, lxy);
        PlaneTail<T, XYLevel<T, OfInverse>> pt{};
        for (unsigned k = 0; k < lxy; ++k) {
            const unsigned l = OfInverse ? k : lxy - 1 - k;
            const Dims n = box_of(l, true, false);
            const Box<T> split = OfInverse ? out : in;
            const Box<T> nat = l ? plane_box(l) : OfInverse ? in : out;
            const Box<T> lo = l + 1 == lxy ? split : plane_box(l + 1);
            const Box<T> from_box = OfInverse ? nat : split, to_box = OfInverse ? split : nat;
            if (l < tail) {
                xy_level<T, OfInverse>(from_box, lo, to_box, n, s);
            } else {
                add_plane(pt, level_of<T, OfInverse>(from_box, lo, to_box, n));
                if (l == (OfInverse ? lxy - 1 : tail)) xy_tail<T, OfInverse>(pt, full.nz, s);
            }
        }
    };
    const Box<T> in = volume(from, full);
    if constexpr (OfInverse) {
        z_phase(in, mid);
        xy_phase(lz ? mid : in, home);
    } else {
        xy_phase(in, mid);
        z_phase(lxy ? mid : in, home);
    }
}

// One group of passes over one box, out of place through tmp0/tmp1, ending in
// `home`; the first pass reads `first` when given (the whole volume's data).
template <class T, bool OfInverse>
void box_passes(T* home, T* tmp0, T* tmp1, Dims full, Dims act, const int* axes, int count, hipStream_t s,
                const T* first = nullptr) {
    const T* src = first ? first : home;
    for (int k = 0; k < count; ++k) {
        T* dst = k == count - 1 ? home : (k & 1 ? tmp1 : tmp0);
        if (dst == src) dst = tmp0;
        adjoint_axis<T, OfInverse>(src, dst, full, act, axes[k], s);
        src = dst;
    }
    if (src != home) {
        const uint64_t total = uint64_t(act.nx) * act.ny * act.nz;
        check_launch_size(total);
        hipLaunchKernelGGL((adjoint_copy<T>), dim3(uint32_t((total + 255) / 256)), dim3(256), 0, s, src, home, full,
                           act, uint32_t(total));
    }
}
}  // namespace

// In place on `data` (full volume), or from `src` into `data` when src is
// given; tmp0/tmp1: two full-volume scratch arrays. Schedules are those of
// transform_forward / transform_inverse, reversed.
template <class T>
void transform_adjoint(T* data, T* tmp0, T* tmp1, Dims full, unsigned lxy, unsigned lz, bool dyadic,
                       bool of_inverse, hipStream_t s, const T* src) {
    if ((lxy || lz) && levels_fit(full, lxy, lz, sizeof(T))) {
        if (of_inverse) adjoint_levels<T, true>(data, src ? src : data, tmp0, tmp1, full, lxy, lz, dyadic, s);
        else adjoint_levels<T, false>(data, src ? src : data, tmp0, tmp1, full, lxy, lz, dyadic, s);
        return;
    }
    // the adjoint of the inverse starts with a pass over the whole volume,
    // which reads src itself; the other schedules start inside a box
    const T* first = src != data && of_inverse && (lxy || lz) ? src : nullptr;
    if (src && src != data && !first)
        hip_check(hipMemcpyAsync(data, src, uint64_t(full.nx) * full.ny * full.nz * sizeof(T),
                                 hipMemcpyDeviceToDevice, s),
                  "copy");
    if (dyadic) {
        Dims sizes[5], act = full;
        for (unsigned l = 0; l < lxy; ++l) {
            sizes[l] = act;
            act = shrink_box(act, true, true);
        }
        if (!of_inverse) {  // forward: levels 0..L-1, axes Y, X, Z -> reversed
            static const int zxy[3] = {2, 0, 1};
            for (int l = int(lxy) - 1; l >= 0; --l) box_passes<T, false>(data, tmp0, tmp1, full, sizes[l], zxy, 3, s);
        } else {  // inverse: levels L-1..0, axes Z, X, Y -> reversed
            static const int yxz[3] = {1, 0, 2};
            for (unsigned l = 0; l < lxy; ++l)
                box_passes<T, true>(data, tmp0, tmp1, full, sizes[l], yxz, 3, s, l == 0 ? first : nullptr);
        }
        return;
    }
    Dims xy[5], zs[5], act = full;
    for (unsigned l = 0; l < lxy; ++l) {
        xy[l] = act;
        act = shrink_box(act, true, false);
    }
    act = full;
    for (unsigned l = 0; l < lz; ++l) {
        zs[l] = act;
        act = shrink_box(act, false, true);
    }
    static const int zonly[1] = {2};
    if (!of_inverse) {  // forward: Z levels 0..lz-1, then XY levels (Y, X) 0..lxy-1 -> reversed
        static const int xy_rev[2] = {0, 1};
        for (int l = int(lxy) - 1; l >= 0; --l) box_passes<T, false>(data, tmp0, tmp1, full, xy[l], xy_rev, 2, s);
        for (int l = int(lz) - 1; l >= 0; --l) box_passes<T, false>(data, tmp0, tmp1, full, zs[l], zonly, 1, s);
    } else {  // inverse: XY levels (X, Y) lxy-1..0, then Z levels lz-1..0 -> reversed
        static const int yx[2] = {1, 0};
        for (unsigned l = 0; l < lz; ++l)
            box_passes<T, true>(data, tmp0, tmp1, full, zs[l], zonly, 1, s, l == 0 ? first : nullptr);
        for (unsigned l = 0; l < lxy; ++l)
            box_passes<T, true>(data, tmp0, tmp1, full, xy[l], yx, 2, s, l == 0 && !lz ? first : nullptr);
    }
}

template void transform_adjoint<float>(float*, float*, float*, Dims, unsigned, unsigned, bool, bool, hipStream_t,
                                       const float*);
template void transform_adjoint<double>(double*, double*, double*, Dims, unsigned, unsigned, bool, bool,
                                        hipStream_t, const double*);

}  // namespace wz
