// Arguments and launchers of the fused per-level lifting kernels (fused.hip).
#pragma once

#include "common.hpp"
#include "windows.hpp"

namespace wz {

template <class T>
struct FwdLevel {
    const T* src;       // level input box (x fastest)
    uint64_t spy, spz;  // its row / plane pitch (elements)
    Dims n;             // level box extents
    T* hi;              // coefficient volume (seven high bands)
    uint64_t hpy, hpz;
    T* lo;              // LLL destination (next level's input box)
    uint64_t lpy, lpz;
    uint32_t sz;        // z segment length (even)
    uint32_t* status;   // non-null: screen the input for non-finite samples
};

enum InvEmit : int {
    kEmitStore = 0,        // write the reconstruction
    kEmitStoreScreen = 1,  // write it and flag non-finite samples
    kEmitRepair = 2,       // no write: native repair records against `orig`
};

template <class T>
struct InvLevel {
    const T* hi;        // coefficient volume (high bands of this level)
    uint32_t hpy, hpz;  // pitches in elements (planes below 4 GiB)
    const T* lo;        // reconstructed LLL box of the coarser level
    uint32_t lpy, lpz;
    Dims n;             // level box extents
    T* out;             // reconstructed level box
    uint32_t opy, opz;  // (also the pitches of `orig`)
    uint32_t sz;        // z segment length (multiple of 16)
    int emit;           // InvEmit
    uint32_t* status;   // screen / strict-bound failures
    const T* orig;      // kEmitRepair: the original field
    double bound;
    float bound_lo;     // float repair emitter: the largest float <= bound
    T q, inv;           // q > 0: high-band loads are quantized and dequantized (repair emitter, store)
    SegList rep;        // kEmitRepair: one segment per workgroup, cap = 64*32*sz
    // kEmitStoreScreen, np > 0: repairs applied as the samples are stored
    // (strictly increasing indices; key table from repair_keys, `keys` words)
    const uint32_t* pidx;
    const T* perr;
    const uint32_t* ptable;
    uint32_t np, keys;
    const DecodeRecord* plan;  // non-null: np and the list's places from this record of `archive`
    const uint8_t* archive;
};

// Repair segments needed by a level-0 inverse with z segment sz.
inline uint64_t inv_segments(Dims n, uint32_t sz) {
    return uint64_t((n.nx + 63) / 64) * ((n.ny + 31) / 32) * ((n.nz + sz - 1) / sz);
}

template <class T>
void launch_fwd_level(const FwdLevel<T>& a, hipStream_t s);
template <class T>
void launch_inv_level(const InvLevel<T>& a, hipStream_t s);
// z segment (a multiple of 16) of the least estimated time over up to `most`
// workgroups per CU, of which `per_cu` run at once. A workgroup streams sz
// planes and 8 of halo, and the level lasts as long as its busiest CU: about
// (sz + 8) times its workgroups, one that runs alone counting 1.2 (nothing
// hides its waits). Against "about 1024 workgroups", the finest level (us):
// forward 512^3 f32 337 -> 275 (1024 workgroups are three at once and then
// one, 512 are two at once), 320^3 f32 107 -> 80, 448x384x400 f32 282 -> 240,
// 320x256x384 f64 181 -> 150.
inline uint32_t best_z_segment(Dims n, uint32_t cus, uint32_t per_cu, uint32_t most) {
    const uint64_t tiles = uint64_t((n.nx + 63) / 64) * ((n.ny + 31) / 32);
    uint32_t best = 0;
    double least = 0;
    for (uint32_t c = most; c; --c) {  // ties: more workgroups
        const uint64_t segs = std::max<uint64_t>(uint64_t(c) * cus / tiles, 1);
        const uint32_t sz = uint32_t(((n.nz + segs - 1) / segs + 15) & ~uint64_t(15));
        const uint64_t per = (tiles * ((n.nz + sz - 1) / sz) + cus - 1) / cus;
        const double cost = (double(sz) + 8) * (double(per) + (per_cu > 1 && per % per_cu == 1 ? 0.2 : 0.0));
        if (!best || cost < least) {
            best = sz;
            least = cost;
        }
    }
    return best;
}
// z segment of the finest level's repair emitter for box n: the tuned segment,
// or, where its tiles outnumber the workgroups the device holds at once, the
// best of those whose tiles do not
template <class T>
uint32_t repair_z_segment(Dims n, uint32_t tuned);

}  // namespace wz
