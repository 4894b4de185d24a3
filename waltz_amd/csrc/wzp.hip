// WZP magnitude/sign stream (cpu/src/wzp_cpu.cpp:769-949) on gfx950.
//
// Stream: [groups x u32 group offset][chunks x 24-bit meta][payload], one chunk
// = 8192 u16 magnitudes, one group = 16 chunks; payload in logical chunk order.
// Chunk payload = magnitude bytes (RZE over BIT_2 planes, or raw LE u16 when
// RZE+2 >= raw size) then the signs of the nonzero magnitudes, LSB first.
//
// Encoder: one 256-thread workgroup (4 wave64s) per chunk. Each thread owns
// 32 magnitudes = one sign word = 64 transformed bytes = 8 bytes of the zero
// bitmap B0 = one byte of B1. All counts are packed two per 32-bit word into
// block-wide scans (wave shuffles + LDS). Each chunk writes its meta, its size
// and its payload into a 16-byte aligned staging slot and ends; no workgroup
// waits for another. A second kernel (pack_chunks) moves the payloads from
// their slots to their final place in logical order and writes the group
// directory; its offsets are sums of the group lengths and chunk sizes.
//
// Decoder: one workgroup per chunk; the chunk offset is the group offset plus
// the sizes of the earlier chunks of its group (from their metas). RZE is
// undone top-down with popcount prefix ranks, then BIT_2, then signs are
// expanded under the nonzero mask. Every read is bounds-checked against the
// stream; inconsistencies raise kCorrupt.
#include <algorithm>
#include <type_traits>

#include "profile.hpp"
#include "sections.hpp"
#include "wzp_encode.hpp"

namespace wz {

template <class Source>
__global__ void __launch_bounds__(256) wzp_encode_kernel(Source src, uint32_t n, uint32_t groups,
                                                         uint8_t* __restrict__ out, uint64_t capacity, WzpScratch w,
                                                         uint32_t* __restrict__ status) {
    encode_chunk(src, blockIdx.x, n, groups, out, capacity, w, status);
}

constexpr uint32_t kPackThreads = 256;
__global__ void __launch_bounds__(kPackThreads) wzp_pack_kernel(uint8_t* __restrict__ out, uint64_t capacity,
                                                                uint32_t chunks, uint32_t groups, WzpScratch w,
                                                                unsigned long long* __restrict__ total,
                                                                uint32_t* __restrict__ status) {
    pack_chunks<kPackThreads, 1>(blockIdx.x, out, capacity, chunks, groups, w, total, status);
}

void wzp_pack(uint32_t n, uint8_t* out, uint64_t capacity, const WzpScratch& w, unsigned long long* total,
              uint32_t* status, hipStream_t s, const SideStream* side) {
    const WzpShape ws = wzp_shape(n);
    hipStream_t ps = s;
    if (side) {
        hip_check(hipEventRecord(side->ready, s), "event record");
        hip_check(hipStreamWaitEvent(side->stream, side->ready, 0), "stream wait");
        ps = side->stream;
    }
    if (ws.chunks) {
        StageClock c("wzp_pack", ps);
        hipLaunchKernelGGL(wzp_pack_kernel, dim3(ws.chunks), dim3(kPackThreads), 0, ps, out, capacity, ws.chunks,
                           ws.groups, w, total, status);
    }
    if (side) hip_check(hipEventRecord(side->done, ps), "event record");
}

void wzp_encode(const uint16_t* mag, const uint32_t* sign, uint32_t n, uint8_t* out, uint64_t capacity, WzpScratch w,
                uint32_t* status, hipStream_t s) {
    const WzpShape ws = wzp_shape(n);
    if (ws.chunks == 0) return;
    hipLaunchKernelGGL(wzp_encode_kernel<MagSource>, dim3(ws.chunks), dim3(kThreads), 0, s, MagSource{mag, sign}, n,
                       ws.groups, out, capacity, w, status);
}

// The write-back box of a fused quantizing encoder.
template <class T>
void check_direct_bricks(Dims d, uint32_t bz) {
    if (!direct_bricks_fit(d.nx, d.ny, d.nz, bz, sizeof(T)))
        throw std::invalid_argument("field does not tile into direct bricks");
}
// f(true_type) for cubes, f(false_type) for the flatter bands (float only)
template <class T, class F>
void of_band(uint32_t bz, F&& f) {
    if constexpr (sizeof(T) == 4) {
        if (bz != 16) return f(std::false_type{});
    }
    f(std::true_type{});
}

template <class T>
void quantize_encode_direct(T* coeff, Dims d, uint32_t bz, double quantum, SideList qo, uint8_t* out,
                            uint64_t capacity, WzpScratch w, uint32_t* status, hipStream_t s, WriteBack wb) {
    check_direct_bricks<T>(d, bz);
    const uint32_t n = d.nx * d.ny * d.nz;
    const WzpShape ws = wzp_shape(n);
    const Dims h = writeback_box(d, wb);
    const DirectBricks g = DirectBricks::of(d, bz);
    const T q = T(quantum), inv = T(1.0 / quantum);
    of_band<T>(bz, [&](auto cube) {
        using Source = BrickSource<T, decltype(cube)::value>;
        hipLaunchKernelGGL((wzp_encode_kernel<Source>), dim3(ws.chunks), dim3(kThreads), 0, s,
                           Source{coeff, g, q, inv, qo, h.nx, h.ny, h.nz}, n, ws.groups, out, capacity, w, status);
    });
}

void check_rank_bricks(Dims d, uint32_t bz, const uint16_t* rank) {
    if (!rank_bricks_fit(d.nx, d.ny, d.nz, bz) || reinterpret_cast<uintptr_t>(rank) % 8)
        throw std::invalid_argument("field does not tile into full bricks");
}

template <class T>
void quantize_encode_ranks(T* coeff, Dims d, uint32_t bz, const uint16_t* rank, double quantum, SideList qo,
                           uint8_t* out, uint64_t capacity, WzpScratch w, uint32_t* status, hipStream_t s,
                           WriteBack wb) {
    check_rank_bricks(d, bz, rank);
    const uint32_t n = d.nx * d.ny * d.nz;
    const WzpShape ws = wzp_shape(n);
    const Dims h = writeback_box(d, wb);
    const RankSource<T> src{coeff, RankBricks{rank, d.nx, d.ny, bz}, T(quantum), T(1.0 / quantum), qo, h.nx, h.ny,
                            h.nz};
    hipLaunchKernelGGL(wzp_encode_kernel<RankSource<T>>, dim3(ws.chunks), dim3(kThreads), 0, s, src, n, ws.groups,
                       out, capacity, w, status);
}

template <class Sink>
__global__ void __launch_bounds__(256, 8) wzp_decode_kernel(const uint8_t* __restrict__ in, uint64_t bytes, uint32_t n,
                                                         uint32_t chunks, uint32_t groups, Sink sink,
                                                         uint32_t* __restrict__ status) {
    decode_chunk(in, bytes, n, chunks, groups, blockIdx.x, sink, status);
}

__global__ void __launch_bounds__(kDirThreads) wzp_directory_kernel(const uint8_t* __restrict__ in, uint64_t bytes,
                                                                   uint32_t n, uint32_t chunks, uint32_t groups,
                                                                   uint32_t* __restrict__ status) {
    __shared__ uint32_t len[kMaxGroups];
    __shared__ uint32_t sh[kDirThreads / 64];
    check_directory(in, bytes, n, chunks, groups, len, sh, status);
}

// Planned decode: the stream size and quantum come from the device record.
__global__ void __launch_bounds__(kDirThreads) wzp_directory_planned_kernel(const uint8_t* __restrict__ in,
                                                                           const DecodeRecord* __restrict__ rec,
                                                                           uint32_t n, uint32_t chunks,
                                                                           uint32_t groups,
                                                                           uint32_t* __restrict__ status) {
    __shared__ uint32_t len[kMaxGroups];
    __shared__ uint32_t sh[kDirThreads / 64];
    if (!rec->ok) return;
    check_directory(in, rec->wzp, n, chunks, groups, len, sh, status);
}

// The same beside the q-outlier patch (workgroups from 1 on), which follows the
// chunk decoders.
constexpr uint32_t kQpatchBlocks = 32;
template <class T>
__global__ void __launch_bounds__(kDirThreads) directory_qpatch_planned_kernel(T* __restrict__ coeff,
                                                                               const uint8_t* __restrict__ archive,
                                                                               const DecodeRecord* __restrict__ rec,
                                                                               uint32_t n, uint32_t chunks,
                                                                               uint32_t groups,
                                                                               uint32_t* __restrict__ status) {
    __shared__ uint32_t len[kMaxGroups];
    __shared__ uint32_t sh[kDirThreads / 64];
    if (!rec->ok) return;
    if (blockIdx.x == 0) {
        check_directory(archive + 32, rec->wzp, n, chunks, groups, len, sh, status);
        return;
    }
    const uint32_t count = rec->nq;
    const auto* idx = reinterpret_cast<const uint32_t*>(archive + rec->qi);
    const auto* val = reinterpret_cast<const uint32_t*>(archive + rec->qv);
    const T q = T(rec->quantum);
    for (uint32_t j = (blockIdx.x - 1) * kDirThreads + threadIdx.x; j < count; j += (gridDim.x - 1) * kDirThreads)
        qpatch_one(coeff, idx, val, j, n, q, status);
}

template <class T, bool Cube>
__global__ void __launch_bounds__(256, 8) wzp_decode_direct_planned_kernel(const uint8_t* __restrict__ in,
                                                                       const DecodeRecord* __restrict__ rec,
                                                                       uint32_t n, uint32_t chunks, uint32_t groups,
                                                                       T* __restrict__ coeff, DirectBricks g,
                                                                       uint32_t* __restrict__ status) {
    if (!rec->ok) return;
    decode_chunk(in, rec->wzp, n, chunks, groups, blockIdx.x, BrickSink<T, Cube>{coeff, g, T(rec->quantum)}, status);
}

template <class T>
__global__ void __launch_bounds__(256, 8) wzp_decode_ranks_planned_kernel(const uint8_t* __restrict__ in,
                                                                      const DecodeRecord* __restrict__ rec,
                                                                      uint32_t n, uint32_t chunks, uint32_t groups,
                                                                      T* __restrict__ coeff, RankBricks g,
                                                                      uint32_t* __restrict__ status) {
    if (!rec->ok) return;
    decode_chunk(in, rec->wzp, n, chunks, groups, blockIdx.x, RankSink<T>{coeff, g, T(rec->quantum)}, status);
}

__global__ void __launch_bounds__(256, 8) wzp_decode_mag_planned_kernel(const uint8_t* __restrict__ in,
                                                                    const DecodeRecord* __restrict__ rec, uint32_t n,
                                                                    uint32_t chunks, uint32_t groups, MagSink sink,
                                                                    uint32_t* __restrict__ status) {
    if (!rec->ok) return;
    decode_chunk(in, rec->wzp, n, chunks, groups, blockIdx.x, sink, status);
}

// A stream's chunk decoders, enqueued on s first (the device starts them as
// soon as the work before them ends), and its directory check, on the side
// stream when given (both only read the stream and report into the status).
template <class Decoders, class Directory>
void stream_decode(uint32_t n, hipStream_t s, const SideStream* side, Decoders decoders, Directory directory) {
    const WzpShape ws = wzp_shape(n);
    if (side) hip_check(hipEventRecord(side->ready, s), "event record");
    if (ws.chunks) decoders(ws);
    hipStream_t ds = s;
    if (side) {
        hip_check(hipStreamWaitEvent(side->stream, side->ready, 0), "stream wait");
        ds = side->stream;
    }
    if (ws.chunks) directory(ws, ds);
    if (side) hip_check(hipEventRecord(side->done, ds), "event record");
}

template <class T>
void decode_dequantize_direct_planned(const uint8_t* in, const DecodeRecord* rec, Dims d, uint32_t bz, T* coeff,
                                      uint32_t* status, hipStream_t s) {
    check_direct_bricks<T>(d, bz);
    const uint32_t n = d.nx * d.ny * d.nz;
    const WzpShape ws = wzp_shape(n);
    if (!ws.chunks) return;
    const DirectBricks g = DirectBricks::of(d, bz);
    of_band<T>(bz, [&](auto cube) {
        hipLaunchKernelGGL((wzp_decode_direct_planned_kernel<T, decltype(cube)::value>), dim3(ws.chunks),
                           dim3(kThreads), 0, s, in, rec, n, ws.chunks, ws.groups, coeff, g, status);
    });
}

template <class T>
void decode_dequantize_ranks_planned(const uint8_t* in, const DecodeRecord* rec, Dims d, uint32_t bz,
                                     const uint16_t* rank, T* coeff, uint32_t* status, hipStream_t s) {
    check_rank_bricks(d, bz, rank);
    const uint32_t n = d.nx * d.ny * d.nz;
    const WzpShape ws = wzp_shape(n);
    if (!ws.chunks) return;
    hipLaunchKernelGGL(wzp_decode_ranks_planned_kernel<T>, dim3(ws.chunks), dim3(kThreads), 0, s, in, rec, n,
                       ws.chunks, ws.groups, coeff, RankBricks{rank, d.nx, d.ny, bz}, status);
}

void wzp_decode_planned(const uint8_t* in, const DecodeRecord* rec, uint32_t n, uint16_t* mag, uint32_t* sign,
                        uint32_t* status, hipStream_t s) {
    const WzpShape ws = wzp_shape(n);
    if (!ws.chunks) return;
    hipLaunchKernelGGL(wzp_decode_mag_planned_kernel, dim3(ws.chunks), dim3(kThreads), 0, s, in, rec, n, ws.chunks,
                       ws.groups, MagSink{mag, sign}, status);
}

void wzp_directory_planned(const uint8_t* in, const DecodeRecord* rec, uint32_t n, uint32_t* status, hipStream_t s) {
    const WzpShape ws = wzp_shape(n);
    if (!ws.chunks) return;
    hipLaunchKernelGGL(wzp_directory_planned_kernel, dim3(1), dim3(kDirThreads), 0, s, in, rec, n, ws.chunks,
                       ws.groups, status);
}

template <class T>
void directory_qoutliers_planned(T* coeff, const uint8_t* archive, const DecodeRecord* rec, uint32_t n,
                                 uint32_t* status, hipStream_t s) {
    const WzpShape ws = wzp_shape(n);
    if (!ws.chunks) return;
    const uint32_t blocks = 1 + std::min(kQpatchBlocks, (n + kDirThreads - 1) / kDirThreads);
    hipLaunchKernelGGL((directory_qpatch_planned_kernel<T>), dim3(blocks), dim3(kDirThreads), 0, s, coeff, archive, rec,
                       n, ws.chunks, ws.groups, status);
}
template void directory_qoutliers_planned<float>(float*, const uint8_t*, const DecodeRecord*, uint32_t, uint32_t*,
                                                 hipStream_t);
template void directory_qoutliers_planned<double>(double*, const uint8_t*, const DecodeRecord*, uint32_t, uint32_t*,
                                                  hipStream_t);

void wzp_decode(const uint8_t* in, uint64_t bytes, uint32_t n, uint16_t* mag, uint32_t* sign, uint32_t* status,
                hipStream_t s, const SideStream* side) {
    if (n && bytes < wzp_shape(n).header) throw std::runtime_error("WZP archive size is outside its valid bounds");
    stream_decode(
        n, s, side,
        [&](const WzpShape& ws) {
            hipLaunchKernelGGL(wzp_decode_kernel<MagSink>, dim3(ws.chunks), dim3(kThreads), 0, s, in, bytes, n,
                               ws.chunks, ws.groups, MagSink{mag, sign}, status);
        },
        [&](const WzpShape& ws, hipStream_t ds) {
            hipLaunchKernelGGL(wzp_directory_kernel, dim3(1), dim3(kDirThreads), 0, ds, in, bytes, n, ws.chunks,
                               ws.groups, status);
        });
}

template <class T>
void decode_dequantize_direct(const uint8_t* in, uint64_t bytes, Dims d, uint32_t bz, double quantum, T* coeff,
                              uint32_t* status, hipStream_t s, const SideStream* side) {
    check_direct_bricks<T>(d, bz);
    const uint32_t n = d.nx * d.ny * d.nz;
    if (bytes < wzp_shape(n).header) throw std::runtime_error("WZP archive size is outside its valid bounds");
    const DirectBricks g = DirectBricks::of(d, bz);
    stream_decode(
        n, s, side,
        [&](const WzpShape& ws) {
            of_band<T>(bz, [&](auto cube) {
                using Sink = BrickSink<T, decltype(cube)::value>;
                hipLaunchKernelGGL((wzp_decode_kernel<Sink>), dim3(ws.chunks), dim3(kThreads), 0, s, in, bytes, n,
                                   ws.chunks, ws.groups, Sink{coeff, g, T(quantum)}, status);
            });
        },
        [&](const WzpShape& ws, hipStream_t ds) {
            hipLaunchKernelGGL(wzp_directory_kernel, dim3(1), dim3(kDirThreads), 0, ds, in, bytes, n, ws.chunks,
                               ws.groups, status);
        });
}

template <class T>
void decode_dequantize_ranks(const uint8_t* in, uint64_t bytes, Dims d, uint32_t bz, const uint16_t* rank,
                             double quantum, T* coeff, uint32_t* status, hipStream_t s, const SideStream* side) {
    check_rank_bricks(d, bz, rank);
    const uint32_t n = d.nx * d.ny * d.nz;
    if (bytes < wzp_shape(n).header) throw std::runtime_error("WZP archive size is outside its valid bounds");
    const RankSink<T> sink{coeff, RankBricks{rank, d.nx, d.ny, bz}, T(quantum)};
    stream_decode(
        n, s, side,
        [&](const WzpShape& ws) {
            hipLaunchKernelGGL(wzp_decode_kernel<RankSink<T>>, dim3(ws.chunks), dim3(kThreads), 0, s, in, bytes, n,
                               ws.chunks, ws.groups, sink, status);
        },
        [&](const WzpShape& ws, hipStream_t ds) {
            hipLaunchKernelGGL(wzp_directory_kernel, dim3(1), dim3(kDirThreads), 0, ds, in, bytes, n, ws.chunks,
                               ws.groups, status);
        });
}

#define WZ_RANKS(T)                                                                                               \
    template void quantize_encode_ranks<T>(T*, Dims, uint32_t, const uint16_t*, double, SideList, uint8_t*,      \
                                           uint64_t, WzpScratch, uint32_t*, hipStream_t, WriteBack);             \
    template void decode_dequantize_ranks<T>(const uint8_t*, uint64_t, Dims, uint32_t, const uint16_t*, double,  \
                                             T*, uint32_t*, hipStream_t, const SideStream*);                       \
    template void decode_dequantize_ranks_planned<T>(const uint8_t*, const DecodeRecord*, Dims, uint32_t,        \
                                                     const uint16_t*, T*, uint32_t*, hipStream_t);
WZ_RANKS(float)
WZ_RANKS(double)
#undef WZ_RANKS

#define WZ_DIRECT(T)                                                                                              \
    template void quantize_encode_direct<T>(T*, Dims, uint32_t, double, SideList, uint8_t*, uint64_t, WzpScratch, \
                                            uint32_t*, hipStream_t, WriteBack);                                   \
    template void decode_dequantize_direct<T>(const uint8_t*, uint64_t, Dims, uint32_t, double, T*, uint32_t*,     \
                                              hipStream_t, const SideStream*);                                    \
    template void decode_dequantize_direct_planned<T>(const uint8_t*, const DecodeRecord*, Dims, uint32_t, T*,     \
                                                      uint32_t*, hipStream_t);
WZ_DIRECT(float)
WZ_DIRECT(double)
#undef WZ_DIRECT

}  // namespace wz
