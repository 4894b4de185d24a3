// The coarsest XY levels of the plane schedule, shared by the transforms and
// their adjoints (Adjoint: the level transposes of xystrip.hpp).
#pragma once

#include "xystrip.hpp"

namespace wz {
namespace {

// The coarsest XY levels of the plane schedule in one launch: a plane's levels
// depend on nothing else, so a workgroup takes a plane through all levels
// whose boxes are at most kPlaneTailSamples, with a barrier between them
// (planes of 128 x 128 still fill the device better as launches of their own).
constexpr uint32_t kPlaneTailSamples = 4096, kPlaneTailWaves = 8;
template <class T, class Level>
struct PlaneTail {
    uint32_t levels;
    Level level[5];  // in launch order
    StripPlan plan[5];  // of one plane
};
template <class T, bool Adjoint>
__global__ void __launch_bounds__(64 * kPlaneTailWaves) plane_tail_forward_kernel(PlaneTail<T, XYForward<T>> a) {
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), z = blockIdx.x;
    for (uint32_t l = 0; l < a.levels; ++l) {
        XYForward<T> xy = a.level[l];
        xy.src += uint64_t(z) * xy.spz;
        xy.hi += uint64_t(z) * xy.hpz;
        xy.lo += uint64_t(z) * xy.lpz;
        xy.n.nz = 1;
        for (uint32_t i = wave; i < a.plan[l].items(); i += kPlaneTailWaves) strip_forward<T, Adjoint>(xy, a.plan[l], i);
        __syncthreads();
    }
}
template <class T, bool Requant, bool Adjoint>
__global__ void __launch_bounds__(64 * kPlaneTailWaves) plane_tail_inverse_kernel(PlaneTail<T, XYInverse<T>> a) {
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), z = blockIdx.x;
    for (uint32_t l = 0; l < a.levels; ++l) {
        XYInverse<T> xy = a.level[l];
        xy.hi += uint64_t(z) * xy.hpz;
        xy.lo += uint64_t(z) * xy.lpz;
        xy.out += uint64_t(z) * xy.opz;
        xy.n.nz = 1;
        for (uint32_t i = wave; i < a.plan[l].items(); i += kPlaneTailWaves)
            strip_inverse<T, Requant, Adjoint>(xy, a.plan[l], i, StripStore<T>{});
        __syncthreads();
    }
}
// First level of that tail (lxy: none; one level alone is launched as usual).
inline unsigned plane_tail_level(Dims full, unsigned lxy) {
    Dims n = full;
    for (unsigned l = 0; l + 1 < lxy; ++l) {
        if (uint64_t(n.nx) * n.ny <= kPlaneTailSamples) return l;
        n = Dims{half_len(n.nx), half_len(n.ny), n.nz};
    }
    return lxy;
}
template <class T, class Level>
void add_plane(PlaneTail<T, Level>& t, const Level& a) {
    Dims n = a.n;
    n.nz = 1;
    t.plan[t.levels] = strip_plan(n, false, kPlaneTailWaves, 16);
    t.level[t.levels++] = a;
}

// Compact XY boxes of the plane schedule's levels >= 1 (every plane), one after
// the other in `scratch`: a launch that takes a plane through several levels
// must not write one level's box where another plane still reads a finer or
// coarser one. Their sum stays below the field (each is at most 4/9 of the one
// before, for extents of at least 2).
template <class T>
T* xy_box(T* scratch, Dims full, unsigned l) {
    Dims n = full;
    for (unsigned k = 1; k < l; ++k) {
        n = Dims{half_len(n.nx), half_len(n.ny), n.nz};
        scratch += uint64_t(n.nx) * n.ny * n.nz;
    }
    return scratch;
}

}  // namespace
}  // namespace wz
