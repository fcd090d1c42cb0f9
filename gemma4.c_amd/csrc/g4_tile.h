// g4_tile.h -- what the matrix-core GEMM kernels share: operand types, the
// XCD-aware tile order, buffer-resource loads and the LDS-only barrier.
#pragma once
#include "g4_device.h"

namespace g4 {
namespace {

typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef _Float16 h4_t __attribute__((ext_vector_type(4)));
typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef float f4_t __attribute__((ext_vector_type(4)));


__device__ __forceinline__ uint32_t h2_bits(h2_t h) { return __builtin_bit_cast(uint32_t, h); }
__device__ __forceinline__ h2_t bits_h2(uint32_t u) { return __builtin_bit_cast(h2_t, u); }

// fp16 of the half-word pattern 0x64XX is 1024 + XX (XX < 256)
constexpr uint32_t kMagic = 0x64646464u;
constexpr uint32_t kSelLo = 0x04010400u;   // bytes (c0, 0x64, c1, 0x64)
constexpr uint32_t kSelHi = 0x04030402u;   // bytes (c2, 0x64, c3, 0x64)

__device__ __forceinline__ float hbits_to_f32(uint32_t h) {
    _Float16 v;
    const uint16_t b = (uint16_t)h;
    __builtin_memcpy(&v, &b, 2);
    return (float)v;
}

// XCD-aware tile order.  Workgroups go to the 8 XCDs round robin by their
// linear id; tile t = (row group t / gy, token group t % gy) is given to id
// so that each XCD takes a contiguous run of tiles, i.e. a few row groups
// with all their token groups: the weights of those rows stay in that XCD's
// L2 while its workgroups stream the activations.  (A bijection on ids for
// any tile count; grid = gx * gy workgroups in x.)
__device__ __forceinline__ void xcd_tile(int gy, int& bx, int& by) {
    const int n = gridDim.x, id = blockIdx.x;
    const int q = n >> 3, r = n & 7, x = id & 7, l = id >> 3;
    const int t = (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + l;
    bx = t / gy;
    by = t - bx * gy;
}

// buffer-resource loads (word 3 of the descriptor: 32-bit data format, the
// value the gfx9 family takes for raw byte-addressed buffers)
constexpr int kBufWord3 = 0x00020000;
__device__ __forceinline__ uint4 buf_load16(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}
__device__ __forceinline__ uint2 buf_load8(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    return __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
}
__device__ __forceinline__ uint32_t buf_load4(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    return __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0);
}

// Workgroup barrier for LDS hand-offs: this wave's LDS operations complete,
// then s_barrier.  __syncthreads() also waits for every outstanding global
// load (its release fence), which would make each block wait for the next
// block's prefetch; here the loads stay in flight across the barrier.  The
// asm is a compiler barrier for memory operations as well.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// s_waitcnt immediate that waits until at most n vector memory operations
// are outstanding (gfx9 encoding: vmcnt bits 3:0 and 15:14; expcnt and
// lgkmcnt left at their maxima, i.e. not waited for)
constexpr int vmcnt_imm(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8); }

// 16 bytes per lane from a buffer straight into LDS at lds + 16 * lane (the
// LDS address is wave-uniform: it goes to M0).  A plain device function: in
// a kernel template's own body the builtin keeps the host pass from
// emitting the kernel's launch stub.
typedef __attribute__((address_space(3))) void lds_void;
__device__ __forceinline__ void buf_load_lds16(__amdgpu_buffer_rsrc_t r, uint8_t* lds, int voff, int soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)lds, 16, voff, soff, 0, 0);
}

bool al16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

}  // namespace
}  // namespace g4
