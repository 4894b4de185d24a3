// X and Y lifting of one level of a stack of planes in registers (no LDS, no
// barrier), shared by the single-field and batched transforms.
//
// A wave owns a strip of a plane and walks it along y, two rows (one sample
// pair) per step. A lane holds one (even, odd) sample pair of its line in x:
// X lifting takes the neighbouring pairs' values from the neighbouring lanes
// (one cross-lane move each), Y lifting streams down the strip with five live
// values per column. So every value is loaded once (strip ends and the
// warm-up rows of a strip's y segment aside), all loads and stores are whole
// row segments, and a sample costs about 9 vector operations for X and 7 for
// Y, well below what memory takes. Every value is the same sequence of
// operations on the same operands as in lift_tile (inverse Y tile 8 folded,
// X unfolded), so the same bits.
//
// Lines of up to 62 pairs, or of exactly 64, take one strip; longer ones
// strips of 62, then 60 pairs with two pairs of halo on each side. Narrow
// lines share a wave: groups of 8, 16 or 32 lanes take consecutive planes.
// Mirroring: lanes past a line's end load the mirrored samples, so two such
// lanes give the last pair its neighbours; at lane 0 of a line, and at the
// last lane of a line of even length that fills its group, the neighbour's
// value is the lane's own (the lifted extension keeps the symmetry).
#pragma once

#include <type_traits>

#include "buffer.hpp"
#include "common.hpp"
#include "fused.hpp"
#include "launch.hpp"
#include "lifting.hpp"
#include "repair.hpp"

namespace wz {

struct StripPlan {
    uint32_t lw;      // log2 of the lanes of one line (3 .. 6)
    uint32_t strips;  // strips of a line
    uint32_t sy;      // rows of a y segment (a multiple of 8)
    uint32_t segs;    // y segments
    uint32_t zgroups; // groups of 64 >> lw planes
    WZ_HD uint64_t items() const { return uint64_t(strips) * segs * zgroups; }  // waves
};
constexpr uint32_t kStripThreads = 256;

// The plan of an nx x ny box of nz planes; `pack`: lines may share a wave
// (false: the planes of a group would not fit one 32-bit window); `want`: the
// waves this box should come to, where it has the rows for them; `least`: the
// shortest segment it is cut to for that.
WZ_HD StripPlan strip_plan(Dims n, bool pack, uint32_t want = 4096, uint32_t least = 32) {
    StripPlan p;
    const uint32_t np = half_len(n.nx);
    auto fits = [&](uint32_t w) { return np + 2 <= w || (np == w && !(n.nx & 1u)); };
    p.lw = 6;
    if (pack)
        while (p.lw > 3 && fits(1u << (p.lw - 1))) --p.lw;
    p.strips = fits(1u << p.lw) ? 1u : 1u + (np - 62u + 59u) / 60u;
    p.zgroups = (n.nz + (64u >> p.lw) - 1) >> (6 - p.lw);
    // long segments (few warm-up rows), halved while the waves are too few to
    // keep memory busy
    p.sy = 128;
    auto waves = [&] { return uint64_t(p.strips) * p.zgroups * ((n.ny + p.sy - 1) / p.sy); };
    while (p.sy > least && waves() < want) p.sy >>= 1;
    if (waves() < want / 4) p.sy = 16;
    p.segs = (n.ny + p.sy - 1) / p.sy;
    return p;
}

// The value of the lane before / after (cross-lane move over the wave), or the
// lane's own at the end of its line.
WZ_D float lane_prev(float v, bool own) {
    const int x = __builtin_bit_cast(int, v);
    const float r = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, x, 0x138, 0xf, 0xf, true));
    return own ? v : r;
}
WZ_D float lane_next(float v, bool own) {
    const int x = __builtin_bit_cast(int, v);
    const float r = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, x, 0x130, 0xf, 0xf, true));
    return own ? v : r;
}
WZ_D double lane_prev(double v, bool own) {
    const int2 x = __builtin_bit_cast(int2, v);
    const int2 r = make_int2(__builtin_amdgcn_update_dpp(0, x.x, 0x138, 0xf, 0xf, true),
                             __builtin_amdgcn_update_dpp(0, x.y, 0x138, 0xf, 0xf, true));
    return own ? v : __builtin_bit_cast(double, r);
}
WZ_D double lane_next(double v, bool own) {
    const int2 x = __builtin_bit_cast(int2, v);
    const int2 r = make_int2(__builtin_amdgcn_update_dpp(0, x.x, 0x130, 0xf, 0xf, true),
                             __builtin_amdgcn_update_dpp(0, x.y, 0x130, 0xf, 0xf, true));
    return own ? v : __builtin_bit_cast(double, r);
}

// Inverse / forward X lifting of a row, one pair per lane.
template <class T>
WZ_D void strip_x_inverse(T& e, T& o, bool first, bool last) {
    using C = Lift<T>;
    const T o0 = o * (-C::k), e0 = e * C::ik;
    const T e1 = fmadd(-C::d, lane_prev(o0, first) + o0, e0);
    const T o2 = fmadd(-C::g, e1 + lane_next(e1, last), o0);
    e = fmadd(-C::b, lane_prev(o2, first) + o2, e1);
    o = fmadd(-C::a, e + lane_next(e, last), o2);
}
template <class T>
WZ_D void strip_x_forward(T& e, T& o, bool first, bool last) {
    using C = Lift<T>;
    const T o1 = fmadd(C::a, e + lane_next(e, last), o);
    const T e2 = fmadd(C::b, lane_prev(o1, first) + o1, e);
    const T o3 = fmadd(C::g, e2 + lane_next(e2, last), o1);
    const T e4 = fmadd(C::d, lane_prev(o3, first) + o3, e2);
    e = e4 * C::k;
    o = o3 * (-C::ik);
}

// A lifting step on a mirrored line adds c (l + r) of a sample's neighbours to
// it. Its transpose adds c (u l + v r): a sample next to an end of the line
// counts the end twice (the end's own step read that sample twice), and an end,
// whose two neighbours are mirror images of each other, counts them once. In
// terms of t += scale c (l' + r'), l' and r' halved or not, so that nothing is
// doubled before it is multiplied: what fits the type before a step and after
// it fits inside it too, as it does without mirroring.
struct MirrorSteps {
    uint32_t two, left, right;  // bit k, for position q0 + k: scale of 2; l, r halved
};
// Bit k: position q0 + k is an end of a line of n >= 2 samples or the mirror
// image of one (up to four samples outside the line, more on shorter lines).
// `images`: line_images(n).
WZ_HD uint32_t line_images(int32_t n) {  // of lines below 9 samples, bit q + 16
    uint32_t m = n < 9 ? 1u << 16 : 0u;  // (by doubling: a remainder a bit cost a plane tail 1 to 2 us)
    for (int k = 0; k < 5; ++k) {
        const uint32_t s = uint32_t(n - 1) << k;
        if (s < 32) m |= m << s | m >> s;
    }
    return m;
}
WZ_HD uint32_t line_ends(int32_t q0, int32_t n, uint32_t images) {
    if (images) return images >> min(uint32_t(q0 + 16), 31u);
    const uint32_t a = uint32_t(-q0), b = uint32_t(n - 1 - q0);
    return (a < 32u ? 1u << a : 0u) | (b < 32u ? 1u << b : 0u);
}
WZ_HD MirrorSteps mirror_steps(uint32_t ends) {
    const uint32_t l = ends << 1, r = ends >> 1;
    return {l | r, ends | (r & ~l), ends | (l & ~r)};
}
// f(steps, true_type) when the stream's step of pair g touches an end, else
// f(steps, false_type); position 2g - 5 is bit 0. One scalar compare, and the
// bits only behind it: taken at every step they were 1 to 4 % of the adjoints
// (IDWT^T 256^3 float32 110 -> 106 us, 30x257x255 56 -> 54).
template <class F>
WZ_D void mirror_stream(int32_t g, int32_t n, uint32_t images, F&& f) {
    // (2g - 5 > 0 and 2g + 1 < n - 1: lines of at most 8 have no such step)
    if (uint32_t(g - 3) < uint32_t(max(n - 7, 0)) / 2) f(MirrorSteps{0, 0, 0}, std::false_type{});
    else f(mirror_steps(line_ends(2 * g - 5, n, images)), std::true_type{});
}
// v 2^e (neither zero nor near the ends of the range), on the exponent: scalar
// arithmetic where both are wave-uniform.
WZ_D float times_power(float v, uint32_t e) {
    return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, v) + (e << 23));
}
WZ_D double times_power(double v, uint32_t e) {
    return __builtin_bit_cast(double, __builtin_bit_cast(uint64_t, v) + (uint64_t(e << 20) << 32));
}
// The step into position k of wave-uniform `m`; Ends: not known to be empty.
template <bool Ends, class T>
WZ_D T mirror_lift(T c, T l, T r, T t, const MirrorSteps& m, int k) {
    if constexpr (!Ends) return fmadd(c, l + r, t);
    auto bit = [k](uint32_t w) { return (w >> k) & 1u; };
    const T fl = times_power(T(1), 0u - bit(m.left)), fr = times_power(T(1), 0u - bit(m.right));
    return fmadd(times_power(c, bit(m.two)), fmadd(l, fl, r * fr), t);
}
// The same of the four steps of a pair's two samples (even: steps into the even
// one) with per-lane positions, kept in registers.
template <class T, bool OfInverse>
struct MirrorLine {
    T l[2], r[2];    // factors of a neighbour, into the even / odd sample
    T c[4];          // coefficients of the steps in their order
    WZ_D static MirrorLine of(int32_t q, int32_t n) {
        using C = Lift<T>;
        MirrorLine a;
        const MirrorSteps m = mirror_steps(line_ends(q - 1, n, line_images(n)));  // (q: bit 1)
        const T plain[4] = {OfInverse ? -C::a : C::d, OfInverse ? -C::b : C::g, OfInverse ? -C::g : C::b,
                            OfInverse ? -C::d : C::a};
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            a.l[p] = (m.left >> (p + 1)) & 1u ? T(0.5) : T(1);
            a.r[p] = (m.right >> (p + 1)) & 1u ? T(0.5) : T(1);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int p = OfInverse ? k & 1 : 1 - (k & 1);  // of the inverse: into the even sample first
            a.c[k] = (m.two >> (p + 1)) & 1u ? T(2) * plain[k] : plain[k];
        }
        return a;
    }
    WZ_D T lift(int k, T left, T right, T t) const {
        const int p = OfInverse ? k & 1 : 1 - (k & 1);
        return fmadd(c[k], fmadd(left, l[p], right * r[p]), t);
    }
};
// The transposed steps of the inverse / forward X lifting (Adjoint in
// strip_forward and strip_inverse).
template <class T>
WZ_D void strip_x_inverse_adjoint(T& e, T& o, bool first, bool last, const MirrorLine<T, true>& m) {
    using C = Lift<T>;
    const T e1 = m.lift(0, lane_prev(o, first), o, e);
    const T o1 = m.lift(1, e1, lane_next(e1, last), o);
    const T e2 = m.lift(2, lane_prev(o1, first), o1, e1);
    const T o2 = m.lift(3, e2, lane_next(e2, last), o1);
    e = e2 * C::ik;
    o = o2 * (-C::k);
}
template <class T>
WZ_D void strip_x_forward_adjoint(T& e, T& o, bool first, bool last, const MirrorLine<T, false>& m) {
    using C = Lift<T>;
    const T e0 = e * C::k, o0 = o * (-C::ik);
    const T o1 = m.lift(0, e0, lane_next(e0, last), o0);
    const T e1 = m.lift(1, lane_prev(o1, first), o1, e0);
    o = m.lift(2, e1, lane_next(e1, last), o1);
    e = m.lift(3, lane_prev(o, first), o, e1);
}

// Two consecutive samples (dword-aligned).
WZ_D void buf_load_pair(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff, float& a, float& b) {
    using F2 = float __attribute__((ext_vector_type(2)));
    const F2 v = __builtin_bit_cast(F2, __builtin_amdgcn_raw_buffer_load_b64(r, int(voff), int(soff), 0));
    a = v.x;
    b = v.y;
}
WZ_D void buf_load_pair(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff, double& a, double& b) {
    using D2 = double __attribute__((ext_vector_type(2)));
    const D2 v = __builtin_bit_cast(D2, __builtin_amdgcn_raw_buffer_load_b128(r, int(voff), int(soff), 0));
    a = v.x;
    b = v.y;
}
WZ_D void buf_store_pair(float a, float b, __amdgpu_buffer_rsrc_t r, uint32_t voff) {
    using F2 = float __attribute__((ext_vector_type(2)));
    using U2 = unsigned __attribute__((ext_vector_type(2)));
    const F2 v = {a, b};
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U2, v), r, int(voff), 0, 0);
}
WZ_D void buf_store_pair(double a, double b, __amdgpu_buffer_rsrc_t r, uint32_t voff) {
    using D2 = double __attribute__((ext_vector_type(2)));
    using U4 = unsigned __attribute__((ext_vector_type(4)));
    const D2 v = {a, b};
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(U4, v), r, int(voff), 0, 0);
}

// A wave's item: its strip, y segment and planes, and each lane's pair.
struct StripItem {
    uint32_t z0, zl;  // first plane, and the lane's plane less it (in range)
    uint32_t ys, blocks;  // first row, blocks of 8 rows
    uint32_t kp;      // the lane's pair in x
    bool own;         // the lane's pair is the strip's to write
    bool first, last; // line ends at this lane's group edges
};
WZ_D StripItem strip_item(const StripPlan& p, Dims n, uint32_t item) {
    StripItem it;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t strip = item % p.strips, r = item / p.strips, seg = r % p.segs, zg = r / p.segs;
    const uint32_t group = lane >> p.lw, w = 1u << p.lw, k = lane & (w - 1u), per = 64u >> p.lw;
    it.z0 = zg * per;
    const uint32_t z = it.z0 + group;
    it.zl = min(z, n.nz - 1u) - it.z0;
    it.ys = seg * p.sy;
    it.blocks = (min(p.sy, n.ny - it.ys) + 7) / 8;
    const uint32_t np = half_len(n.nx);
    const uint32_t b0 = strip ? 62u + 60u * (strip - 1u) : 0u;
    const uint32_t b1 = p.strips == 1 ? np : min(np, strip ? b0 + 60u : 62u);
    it.kp = (strip ? b0 - 2u : 0u) + k;
    it.own = z < n.nz && it.kp >= b0 && it.kp < b1;
    it.first = k == 0;
    it.last = k == w - 1u;
    return it;
}

// What becomes of an inverse strip's samples. box(): extents that are kept;
// fetch(y): what rows y and y + 1 need is loaded ahead; put(): rows y, y + 1 of
// the lane's two columns, `both` / `half`: the lane keeps its two samples, or
// the first only; in0, in1: the rows are kept (wave-uniform); `wo`, `ov`,
// `orow`: the destination's window, the lane's offset and the row pitch.
template <class T>
struct StripStore {
    WZ_D Dims box(Dims n) const { return n; }
    WZ_D void fetch(uint32_t) {}
    WZ_D void put(uint32_t y, const T (&r0)[2], const T (&r1)[2], bool both, bool half, bool in0, bool in1, bool odd,
                  __amdgpu_buffer_rsrc_t wo, uint32_t ov, uint32_t orow) {
        // lanes and rows outside go past the window's range (dropped)
        const uint32_t at = ov + y * orow;
        buf_store_pair(r0[0], r0[1], wo, both && in0 ? at : kOutside);
        buf_store_pair(r1[0], r1[1], wo, both && in1 ? at + orow : kOutside);
        if (odd) {  // the last sample of an odd line
            buf_store(r0[0], wo, half && in0 ? at : kOutside);
            buf_store(r1[0], wo, half && in1 ? at + orow : kOutside);
        }
    }
};
// The same with a non-finite screen, clipped to an output frame, or a hole's
// fill value instead of the samples.
template <class T>
struct StripOutput {
    Dims frame;
    bool hole;
    T fill;
    bool finite = true;
    WZ_D Dims box(Dims) const { return frame; }
    WZ_D void fetch(uint32_t) {}
    WZ_D void put(uint32_t y, T (&r0)[2], T (&r1)[2], bool both, bool half, bool in0, bool in1, bool odd,
                  __amdgpu_buffer_rsrc_t wo, uint32_t ov, uint32_t orow) {
        auto value = [&](T& v, bool kept) {
            if (hole) v = fill;
            else finite = finite && (finite_value(v) || !kept);
        };
        value(r0[0], (both || half) && in0);
        value(r0[1], both && in0);
        value(r1[0], (both || half) && in1);
        value(r1[1], both && in1);
        StripStore<T>{}.put(y, r0, r1, both, half, in0, in1, odd, wo, ov, orow);
    }
};
// Compared with the originals (the destination's window and pitches are
// theirs) instead of stored: flag bits (of a cleared bitmap: rows share words)
// and records in the wave's own segment of `cap` entries, counted in a scalar.
template <class T>
struct StripRepair {
    WaveRepair<T> r;
    uint32_t segment;     // the wave's item
    uint32_t row0, nx;    // sample index of the lane's pair in row 0; samples per row
    __amdgpu_buffer_rsrc_t wo;
    uint32_t ov, orow;
    T ref[2][2] = {};
    uint32_t fill = 0;
    bool ok = true;
    WZ_D Dims box(Dims n) const { return n; }
    WZ_D void fetch(uint32_t y) {
        buf_load_pair(wo, ov + y * orow, 0u, ref[0][0], ref[0][1]);
        buf_load_pair(wo, ov + (y + 1) * orow, 0u, ref[1][0], ref[1][1]);
    }
    WZ_D void put(uint32_t y, const T (&r0)[2], const T (&r1)[2], bool both, bool half, bool in0, bool in1, bool,
                  __amdgpu_buffer_rsrc_t, uint32_t, uint32_t) {
        const bool kept[2] = {both || half, both};
        const unsigned long long km[2] = {__ballot(kept[0]), __ballot(kept[1])};
        uint32_t* const index = r.rep.index + uint64_t(segment) * r.rep.cap;
        T* const payload = static_cast<T*>(r.rep.payload) + uint64_t(segment) * r.rep.cap;
        const uint32_t lane = threadIdx.x & 63u;
#pragma unroll
        for (int row = 0; row < 2; ++row) {
            if (!(row ? in1 : in0)) continue;  // (wave-uniform)
            const T(&v)[2] = row ? r1 : r0;
            const uint32_t at = row0 + (y + uint32_t(row)) * nx;
            unsigned long long m[2];
#pragma unroll
            for (int c = 0; c < 2; ++c) m[c] = repair_mask<T>(v[c], ref[row][c], kept[c], km[c], r, &ok);
            const bool p0 = (m[0] >> lane) & 1ull, p1 = (m[1] >> lane) & 1ull;
            if (p0 || p1) {
                const uint32_t s = at & 31u, bits = uint32_t(p0) | uint32_t(p1) << 1;
                atomicOr(&r.rep.bitmap[at >> 5], bits << s);
                if (s == 31 && p1) atomicOr(&r.rep.bitmap[(at >> 5) + 1], 1u);
            }
            const unsigned long long below = (1ull << lane) - 1ull;
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                if (c ? p1 : p0) {
                    const uint32_t k = fill + uint32_t(__popcll(m[c] & below));
                    index[k] = at + uint32_t(c);
                    payload[k] = v[c] - ref[row][c];
                }
                fill += uint32_t(__popcll(m[c]));
            }
        }
    }
};

template <class T>
struct XYInverse {
    const T* hi;  // the level's coefficients outside its low box
    uint64_t hpy, hpz;
    const T* lo;  // its low box [0, ceil(nx/2)) x [0, ceil(ny/2)): the coarser reconstruction
    uint64_t lpy, lpz;
    T* out;  // the level's reconstruction (natural layout)
    uint64_t opy, opz;
    Dims n;  // level box: nx x ny, every plane
    // q > 0: the coefficients hold unquantized values, quantized and
    // dequantized as they load (the low box too when lo_coeff: the coarsest
    // level, whose low box is the coefficient volume's)
    T q, inv;
    uint32_t lo_coeff;
};

// One item of an inverse level (nx, ny >= 2): the step of pair g loads pair
// g + 2 and emits rows 2 (g - 2) and 2 (g - 2) + 1; the segment's first four
// steps only warm the Y pipeline up. Four steps are one block (the fold phases
// of the Y tile of 8 rows are then fixed). Adjoint: the transpose of the
// forward level instead, whose input is the split gradient.
template <class T, bool Requant, bool Adjoint = false, class Output>
WZ_D void strip_inverse(const XYInverse<T>& a, const StripPlan& p, uint32_t item, Output&& out) {
    using C = Lift<T>;
    constexpr uint32_t S = sizeof(T);
    const Dims n = a.n;
    const StripItem it = strip_item(p, n, item);
    const uint32_t hy = half_len(n.ny);
    const int32_t ny = int32_t(n.ny);
    const uint32_t ce = split_pos(int32_t(2 * it.kp), n.nx), co = split_pos(int32_t(2 * it.kp + 1), n.nx);
    const auto wh = window(a.hi + uint64_t(it.z0) * a.hpz), wl = window(a.lo + uint64_t(it.z0) * a.lpz);
    const uint32_t hrow = uint32_t(a.hpy) * S, lrow = uint32_t(a.lpy) * S, orow = uint32_t(a.opy) * S;
    const uint32_t lv = (it.zl * uint32_t(a.lpz) + ce) * S, hv = it.zl * uint32_t(a.hpz) * S;
    const uint32_t he = hv + ce * S, ho = hv + co * S;
    const auto wo = window_n(a.out + uint64_t(it.z0) * a.opz,
                             uint32_t((uint64_t(min(64u >> p.lw, n.nz - it.z0) - 1u) * a.opz +
                                       uint64_t(n.ny - 1u) * a.opy + n.nx) * S));
    const uint32_t ov = (it.zl * uint32_t(a.opz) + 2 * it.kp) * S;
    const Dims c = out.box(n);
    const bool here = it.own && it.z0 + (threadIdx.x & 63u) / (1u << p.lw) < c.nz;
    const bool both = here && 2 * it.kp + 1 < c.nx, half = here && 2 * it.kp + 1 == c.nx;
    if constexpr (std::is_same_v<std::decay_t<Output>, StripRepair<T>>) {
        out.segment = item;
        out.nx = n.nx;
        out.row0 = (it.z0 + it.zl) * n.nx * n.ny + 2 * it.kp;
        out.wo = wo;
        out.ov = ov;
        out.orow = orow;
    }
    auto load = [&](int32_t g, T (&v)[4]) {  // pair g of rows: (low, high) of its even and of its odd row
        const uint32_t se = uint32_t(pair_even(g, ny)), so = hy + uint32_t(pair_odd(g, ny));
        v[0] = buf_load_at(T(0), wl, lv, se * lrow);
        v[1] = buf_load_at(T(0), wh, ho, se * hrow);
        v[2] = buf_load_at(T(0), wh, he, so * hrow);
        v[3] = buf_load_at(T(0), wh, ho, so * hrow);
    };
    T OS[2], EA[2], OB[2], EC[2], SF[2];  // Y state, as the fused level's Z synthesis
#pragma unroll
    for (int c = 0; c < 2; ++c) OS[c] = EA[c] = OB[c] = EC[c] = SF[c] = T(0);
    std::conditional_t<Adjoint, MirrorLine<T, false>, int> line{};
    if constexpr (Adjoint) line = MirrorLine<T, false>::of(int32_t(2 * it.kp), int32_t(n.nx));
    [[maybe_unused]] const uint32_t images = Adjoint ? line_images(ny) : 0u;
    T buf[4][4];
    int32_t g = int32_t(it.ys / 2) - 2;
    load(g, buf[0]);
    load(g + 1, buf[1]);
    auto block = [&](auto emit_c) {
        constexpr bool emit = decltype(emit_c)::value;
#pragma unroll
        for (int u = 0; u < 4; ++u, ++g) {
            load(g + 2, buf[(u + 2) & 3]);
            if constexpr (emit) out.fetch(2 * uint32_t(g - 2));
            T(&v)[4] = buf[u];
            if constexpr (Requant) {
                if (a.lo_coeff) v[0] = requantize<T>(v[0], a.q, a.inv);
#pragma unroll
                for (int i = 1; i < 4; ++i) v[i] = requantize<T>(v[i], a.q, a.inv);
            }
            T re[2], ro[2];
            if constexpr (Adjoint) {
                strip_x_forward_adjoint(v[0], v[1], it.first, it.last, line);
                strip_x_forward_adjoint(v[2], v[3], it.first, it.last, line);
                mirror_stream(g, ny, images, [&](const MirrorSteps& m, auto ends_c) {
                    constexpr bool ends = decltype(ends_c)::value;
#pragma unroll
                    for (int c = 0; c < 2; ++c) {  // (the forward pipeline's states: O, O1, E2, O3, E)
                        const T ev = v[c] * C::k, odd = v[2 + c] * (-C::ik);
                        const T o1 = mirror_lift<ends>(C::d, SF[c], ev, OS[c], m, 4);
                        const T e2 = mirror_lift<ends>(C::g, EA[c], o1, SF[c], m, 3);
                        const T o3 = mirror_lift<ends>(C::b, OB[c], e2, EA[c], m, 2);
                        re[c] = mirror_lift<ends>(C::a, EC[c], o3, OB[c], m, 1);
                        ro[c] = o3;
                        SF[c] = ev;
                        OS[c] = odd;
                        EA[c] = o1;
                        OB[c] = e2;
                        EC[c] = o3;
                    }
                });
            } else {
                strip_x_inverse(v[0], v[1], it.first, it.last);
                strip_x_inverse(v[2], v[3], it.first, it.last);
                const int phase = (u + 2) & 3;
#pragma unroll
                for (int c = 0; c < 2; ++c) {  // the pair's columns
                    const T oraw = v[2 + c];
                    const T es = v[c] * C::ik, os = oraw * (-C::k);
                    const T eA = fmadd(-C::d, OS[c] + os, es);
                    const T oB = fmadd(-C::g, EA[c] + eA, OS[c]);
                    const T eC = fmadd(-C::b, OB[c] + oB, EA[c]);
                    re[c] = EC[c];
                    ro[c] = fmadd(-C::a, EC[c] + eC, OB[c]);
                    if (phase == 3) {  // g = B - 1: fold of tile B's first pair
                        SF[c] = fmadd(-C::d, fmadd(SF[c], -C::k, os), es);
                    } else if (phase == 0) {
                        SF[c] = fmadd(-C::g, SF[c] + eA, OS[c]);
                    } else if (phase == 1) {  // and the tile before's last sample
                        SF[c] = fmadd(-C::b, SF[c] + oB, EA[c]);
                        const T eAe = fmadd(-C::d, fmadd(oraw, -C::k, OS[c]), es);
                        const T oBe = fmadd(-C::g, EA[c] + eAe, OS[c]);
                        const T eCe = fmadd(-C::b, OB[c] + oBe, EA[c]);
                        ro[c] = fmadd(-C::a, EC[c] + eCe, OB[c]);
                    } else {  // g = B + 2: tile B's first two samples; o_raw[B' - 2] for the next fold
                        re[c] = SF[c];
                        ro[c] = fmadd(-C::a, SF[c] + eC, OB[c]);
                        SF[c] = oraw;
                    }
                    OS[c] = os;
                    EA[c] = eA;
                    OB[c] = oB;
                    EC[c] = eC;
                }
            }
            if constexpr (emit) {
                const uint32_t y = 2 * uint32_t(g - 2);
                out.put(y, re, ro, both, half, y < c.ny, y + 1 < c.ny, (c.nx & 1u) != 0, wo, ov, orow);
            }
        }
    };
    block(std::false_type{});
    for (uint32_t b = 0; b < it.blocks; ++b) block(std::true_type{});
    if constexpr (std::is_same_v<std::decay_t<Output>, StripRepair<T>>) {
        if ((threadIdx.x & 63u) == 0) out.r.rep.count[item] = out.fill;
    }
}
// Record slots of one item of the repair form.
WZ_HD uint32_t strip_repair_cap(const StripPlan& p) { return p.sy * 128u; }

template <class T>
struct XYForward {
    const T* src;  // the level's input (natural layout)
    uint64_t spy, spz;
    T* hi;  // where the three high bands go
    uint64_t hpy, hpz;
    T* lo;  // where the low band [0, ceil(nx/2)) x [0, ceil(ny/2)) goes
    uint64_t lpy, lpz;
    Dims n;
    uint32_t* status;  // non-null: screen the input for non-finite samples
};

// One item of a forward level (nx, ny >= 2): the step of row pair g loads pair
// g + 2 and emits the low and high row g - 2 of the split. Adjoint: the
// transpose of the inverse level instead, whose input is the gradient of the
// samples. Wide: planes past one window, every row through its own (lines do not
// share a wave then; 33000 x 33000 float: all levels 3.0 ms, as axis passes 10.8).
template <class T, bool Adjoint = false, bool Wide = false>
WZ_D void strip_forward(const XYForward<T>& a, const StripPlan& p, uint32_t item) {
    using C = Lift<T>;
    constexpr uint32_t S = sizeof(T);
    const Dims n = a.n;
    const StripItem it = strip_item(p, n, item);
    const uint32_t hx = half_len(n.nx), hy = half_len(n.ny);
    const int32_t ny = int32_t(n.ny);
    // the pair's two samples are neighbours also where they are mirrored, then
    // in the other order
    const uint32_t xe = reflect_pos(int32_t(2 * it.kp), n.nx), xo = reflect_pos(int32_t(2 * it.kp + 1), n.nx);
    const bool swap = xo < xe;
    const auto ws = window(a.src + uint64_t(it.z0) * a.spz);
    const uint32_t sv = (it.zl * uint32_t(a.spz) + min(xe, xo)) * S, srow = uint32_t(a.spy) * S;
    const uint32_t planes = min(64u >> p.lw, n.nz - it.z0) - 1u;
    const auto wl = window_n(a.lo + uint64_t(it.z0) * a.lpz,
                             uint32_t((uint64_t(planes) * a.lpz + uint64_t(hy - 1u) * a.lpy + hx) * S));
    const auto wh = window_n(a.hi + uint64_t(it.z0) * a.hpz,
                             uint32_t((uint64_t(planes) * a.hpz + uint64_t(n.ny - 1u) * a.hpy + n.nx) * S));
    const uint32_t hrow = uint32_t(a.hpy) * S, lrow = uint32_t(a.lpy) * S;
    const uint32_t lv = (it.zl * uint32_t(a.lpz) + it.kp) * S, hv = (it.zl * uint32_t(a.hpz) + it.kp) * S;
    const bool odd = it.own && 2 * it.kp + 1 < n.nx;
    bool ok = true;
    auto load_row = [&](uint32_t row, T& v0, T& v1) {
        if constexpr (Wide)
            buf_load_pair(window(a.src + uint64_t(it.z0) * a.spz + uint64_t(row) * a.spy), min(xe, xo) * S, 0u, v0, v1);
        else
            buf_load_pair(ws, sv, row * srow, v0, v1);
    };
    auto load = [&](int32_t g, T (&v)[4]) {  // pair g of rows, two samples of each
        load_row(uint32_t(2 * pair_even(g, ny)), v[0], v[1]);
        load_row(uint32_t(2 * pair_odd(g, ny) + 1), v[2], v[3]);
    };
    T E[2], O[2], O1[2], E2[2], O3[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) E[c] = O[c] = O1[c] = E2[c] = O3[c] = T(0);
    std::conditional_t<Adjoint, MirrorLine<T, true>, int> line{};
    if constexpr (Adjoint) line = MirrorLine<T, true>::of(int32_t(2 * it.kp), int32_t(n.nx));
    [[maybe_unused]] const uint32_t images = Adjoint ? line_images(ny) : 0u;
    T buf[4][4];
    int32_t g = int32_t(it.ys / 2) - 2;
    load(g, buf[0]);
    load(g + 1, buf[1]);
    auto block = [&](auto emit_c) {
        constexpr bool emit = decltype(emit_c)::value;
#pragma unroll
        for (int u = 0; u < 4; ++u, ++g) {
            load(g + 2, buf[(u + 2) & 3]);
            const T(&v)[4] = buf[u];
            if (a.status) {  // input screen (cpu/src/codec.cpp:183)
#pragma unroll
                for (int i = 0; i < 4; ++i) ok = ok && finite_value(v[i]);
            }
            T le[2], hi[2];  // the two columns of the low and of the high row
            if constexpr (Adjoint) {
                mirror_stream(g, ny, images, [&](const MirrorSteps& m, auto ends_c) {
                    constexpr bool ends = decltype(ends_c)::value;
#pragma unroll
                    for (int c = 0; c < 2; ++c) {  // (the inverse pipeline's states: OS, EA, OB, EC)
                        const bool other = (c != 0) != swap;
                        const T ev = other ? v[1] : v[0], ov = other ? v[3] : v[2];
                        const T eA = mirror_lift<ends>(-C::a, O[c], ov, ev, m, 5);
                        const T oB = mirror_lift<ends>(-C::b, O1[c], eA, O[c], m, 4);
                        const T eC = mirror_lift<ends>(-C::g, E2[c], oB, O1[c], m, 3);
                        le[c] = O3[c] * C::ik;
                        hi[c] = mirror_lift<ends>(-C::d, O3[c], eC, E2[c], m, 2) * (-C::k);
                        O[c] = ov;
                        O1[c] = eA;
                        E2[c] = oB;
                        O3[c] = eC;
                    }
                });
            } else {
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    const bool other = (c != 0) != swap;
                    const T ev = other ? v[1] : v[0], ov = other ? v[3] : v[2];
                    const T o1 = fmadd(C::a, E[c] + ev, O[c]);
                    const T e2 = fmadd(C::b, O1[c] + o1, E[c]);
                    const T o3 = fmadd(C::g, E2[c] + e2, O1[c]);
                    const T e4 = fmadd(C::d, O3[c] + o3, E2[c]);
                    le[c] = e4 * C::k;
                    hi[c] = o3 * (-C::ik);
                    E[c] = ev;
                    O[c] = ov;
                    O1[c] = o1;
                    E2[c] = e2;
                    O3[c] = o3;
                }
            }
            if constexpr (emit) {
                const uint32_t iy = uint32_t(g - 2);
                if constexpr (Adjoint) {
                    strip_x_inverse_adjoint(le[0], le[1], it.first, it.last, line);
                    strip_x_inverse_adjoint(hi[0], hi[1], it.first, it.last, line);
                } else {
                    strip_x_forward(le[0], le[1], it.first, it.last);
                    strip_x_forward(hi[0], hi[1], it.first, it.last);
                }
                const bool low = 2 * iy < n.ny, high = 2 * iy + 1 < n.ny;
                if constexpr (Wide) {
                    T* const rows = a.hi + uint64_t(it.z0) * a.hpz;
                    const auto ll = window_n(a.lo + uint64_t(it.z0) * a.lpz + uint64_t(iy) * a.lpy, hx * S);
                    const auto lh = window_n(rows + uint64_t(iy) * a.hpy, n.nx * S);
                    const auto hh = window_n(rows + uint64_t(hy + iy) * a.hpy, n.nx * S);
                    const uint32_t x = it.kp * S;
                    buf_store(le[0], ll, it.own && low ? x : kOutside);
                    buf_store(le[1], lh, odd && low ? x + hx * S : kOutside);
                    buf_store(hi[0], hh, it.own && high ? x : kOutside);
                    buf_store(hi[1], hh, odd && high ? x + hx * S : kOutside);
                    continue;
                }
                const uint32_t at = hv + iy * hrow, up = hv + (hy + iy) * hrow;
                buf_store(le[0], wl, it.own && low ? lv + iy * lrow : kOutside);
                buf_store(le[1], wh, odd && low ? at + hx * S : kOutside);
                buf_store(hi[0], wh, it.own && high ? up : kOutside);
                buf_store(hi[1], wh, odd && high ? up + hx * S : kOutside);
            }
        }
    };
    block(std::false_type{});
    for (uint32_t b = 0; b < it.blocks; ++b) block(std::true_type{});
    if (a.status && __ballot(!ok) && (threadIdx.x & 63u) == 0) atomicOr(a.status, uint32_t(kNonFiniteInput));
}

// One XY level (of the plane schedule, or of a dyadic level that runs as
// passes) per launch, four strips of planes per workgroup. Consecutive items
// go to one XCD (workgroups are dealt to the eight XCDs in turn), so that
// neighbours' halos and warm-up rows meet in its L2.
WZ_D bool strip_of_wave(const StripPlan& p, uint32_t& item) {
    const uint32_t total = uint32_t(p.items()), groups = (total + 3) / 4, per = (groups + 7) / 8;
    const uint32_t id = (blockIdx.x & 7u) * per + (blockIdx.x >> 3);
    item = 4 * id + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    return id < groups && item < total;
}
inline uint32_t strip_blocks(const StripPlan& p) {
    const uint64_t groups = (p.items() + 3) / 4, blocks = 8 * ((groups + 7) / 8);
    check_launch_size(blocks * kStripThreads);
    return uint32_t(blocks);
}
// Whether every XY level of an nx x ny plane runs as strips: no line of one
// sample, and a plane inside one 32-bit window.
inline bool strip_lines_fit(Dims n, unsigned levels) { return lines_fit(n.nx, levels) && lines_fit(n.ny, levels); }
inline bool strips_fit(Dims n, uint64_t pitch, uint64_t rows, unsigned levels, unsigned width) {
    return strip_lines_fit(n, levels) && fused_plane_fits(pitch, rows, width);
}
// Lines share a wave only while the planes of a group (at most eight) share a
// window.
inline bool strips_pack(uint64_t plane, unsigned width) { return fused_plane_fits(8 * plane, 1, width); }

}  // namespace wz
