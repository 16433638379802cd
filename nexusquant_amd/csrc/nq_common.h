// Shared device helpers and host error plumbing for the gfx950 kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include "../../include/nexusquant_amd.h"

namespace nq {

// ----------------------------------------------------------------- host ----

void set_error(const char* fmt, ...);

#define NQ_CHECK_ARG(cond, ...)            \
    do {                                   \
        if (!(cond)) {                     \
            ::nq::set_error(__VA_ARGS__);  \
            return NQ_EINVAL;              \
        }                                  \
    } while (0)

// A dispatch's grid size is a 32-bit count of work-items per dimension, so a
// launch of `threads`-wide blocks takes at most this many blocks in one.
constexpr uint64_t max_blocks(uint32_t threads) { return 0xffffffffull / threads; }

#define NQ_CHECK_HIP(expr)                                                   \
    do {                                                                     \
        hipError_t _e = (expr);                                              \
        if (_e != hipSuccess) {                                              \
            ::nq::set_error("%s: %s", #expr, hipGetErrorString(_e));         \
            return NQ_EHIP;                                                  \
        }                                                                    \
    } while (0)

// Address tables of a launch.  A table is an array of tensor base addresses,
// usually in device memory; a pointer with its low bit set (NQ_HOST_ARRAY)
// names a host array instead, whose entries travel inside the kernel's
// arguments: no copy, and no buffer that must outlive the launch.  `inl` is a
// member of the kernel's first argument, struct A; the kernel gets the byte
// offset of the table in its argument segment (never 0, below 4096) in the
// pointer's place and resolves either form with table().
// Measured: staging the addresses of a one-tensor launch through a pinned ring
// (copy, event) cost 11 of 27 us of host time and a copy on the stream.
constexpr int kInlineTabs = NQ_MAX_HOST_ADDRESSES;
struct InlineTabs {
    uint64_t a[kInlineTabs];
};

struct TableSet {
    InlineTabs& inl;
    size_t offset;  // of inl in the kernel's arguments
    int64_t used = 0;
    bool ok = true;  // false: more addresses than the arguments hold

    const uint64_t* take(const uint64_t* p, int64_t n) {
        const uintptr_t v = reinterpret_cast<uintptr_t>(p);
        if (!(v & 1u)) return p;
        if (used + n > kInlineTabs) {
            ok = false;
            return nullptr;
        }
        memcpy(inl.a + used, reinterpret_cast<const uint64_t*>(v - 1), (size_t)n * sizeof(uint64_t));
        const size_t at = offset + (size_t)used * sizeof(uint64_t);
        used += n;
        return reinterpret_cast<const uint64_t*>(at);
    }
};

#define NQ_CHECK_TABLES(set, who) \
    NQ_CHECK_ARG((set).ok, "%s: host arrays hold at most %d addresses a call", who, ::nq::kInlineTabs)

// --------------------------------------------------------------- device ----

// A table's entries: constant for the kernel, so uniform lookups are scalar loads.
typedef const __attribute__((address_space(4))) uint64_t* tab_t;
__device__ __forceinline__ tab_t table(const uint64_t* p) {
    uint64_t a = (uint64_t)p;
    if (a - 1u < 4095u) a += (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
    return (tab_t)a;
}

// Quad (4-lane) permutes through DPP.  Encoded as quad_perm selectors.
constexpr int kQuadXor1 = 0xB1;  // [1,0,3,2]
constexpr int kQuadXor2 = 0x4E;  // [2,3,0,1]

template <int CTRL>
__device__ __forceinline__ float dpp_f32(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, true);
}

__device__ __forceinline__ float bf16_bits_to_f32(uint32_t bits16) {
    return __builtin_bit_cast(float, bits16 << 16);
}
__device__ __forceinline__ float f16_bits_to_f32(uint32_t bits16) {
    return __half2float(__builtin_bit_cast(__half, (unsigned short)bits16));
}
__device__ __forceinline__ uint32_t f32_to_f16_bits(float f) {
    return (uint32_t)__builtin_bit_cast(unsigned short, __float2half_rn(f));
}

}  // namespace nq
