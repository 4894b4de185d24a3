// Raw buffer loads and stores, shared by the fused level and column kernels.
#pragma once

#include "common.hpp"

namespace wz {

// Raw buffer access with a wave-uniform base (a 4 GiB window: stride 0, no
// range limit, dword data format) and a 32-bit per-lane byte offset: no
// per-lane 64-bit address arithmetic.
WZ_D __amdgpu_buffer_rsrc_t window(const void* base) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, -1, 0x00020000);
}
// The same with a byte range: loads beyond it read 0, stores beyond it are
// dropped (how the kernels mask rows and lanes without branching, which keeps
// every step's memory operations and so the memory-counter waits the same).
WZ_D __amdgpu_buffer_rsrc_t window_n(const void* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, int(bytes), 0x00020000);
}
constexpr uint32_t kOutside = 0xFFFFFFF0u;  // a byte offset beyond every window_n range
template <class T>
WZ_D T buf_load(__amdgpu_buffer_rsrc_t r, uint32_t off);
template <>
WZ_D float buf_load<float>(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, int(off), 0, 0));
}
template <>
WZ_D double buf_load<double>(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, int(off), 0, 0));
}
// Streaming (non-temporal) load of data read exactly once (the repair
// emitter's originals), so it does not evict the coefficient lines that
// neighbouring tiles' halos read again.
WZ_D float buf_load_nt(float, __amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, int(off), 0, 2));
}
WZ_D double buf_load_nt(double, __amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, int(off), 0, 2));
}
// Streaming (non-temporal) stores of a level's output: they would otherwise
// evict the input lines that neighbouring tiles' halos read again from L2.
WZ_D void buf_store_nt(float v, __amdgpu_buffer_rsrc_t r, uint32_t off) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, int(off), 0, 2);
}
WZ_D void buf_store_nt(double v, __amdgpu_buffer_rsrc_t r, uint32_t off) {
    using U2 = unsigned __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U2, v), r, int(off), 0, 2);
}
WZ_D void buf_store(float v, __amdgpu_buffer_rsrc_t r, uint32_t off) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, int(off), 0, 0);
}
WZ_D void buf_store(double v, __amdgpu_buffer_rsrc_t r, uint32_t off) {
    using U2 = unsigned __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U2, v), r, int(off), 0, 0);
}

// The same with a wave-uniform byte offset added by the instruction (soff), so
// that rows at scalar places cost no vector arithmetic.
WZ_D float buf_load_at(float, __amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, int(voff), int(soff), 0));
}
WZ_D double buf_load_at(double, __amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, int(voff), int(soff), 0));
}
// (read exactly once: non-temporal, as buf_load_nt)
WZ_D float buf_load_at_nt(float, __amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, int(voff), int(soff), 2));
}
WZ_D double buf_load_at_nt(double, __amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, int(voff), int(soff), 2));
}
WZ_D void buf_store_at(float v, __amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, int(voff), int(soff), 0);
}
WZ_D void buf_store_at(double v, __amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    using U2 = unsigned __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U2, v), r, int(voff), int(soff), 0);
}

}  // namespace wz
