// plane_buffer.hpp -- buffer loads and stores of one z plane.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace scafes {

// Buffer access to one z plane: a wave-uniform resource (base = the plane's
// first memAll element, range = the in-plane extent incl. ghost planes below
// it) plus a 32-bit per-thread byte offset; the hardware range check returns
// 0 for, and drops, accesses beyond the range.
using Rsrc = __amdgpu_buffer_rsrc_t;
constexpr int kRsrcWord3 = 0x00020000;  // gfx9 family: 32-bit data format, raw (stride 0) buffer

__device__ inline Rsrc plane_rsrc(const char* plane, uint32_t range)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(plane), (short)0, (int)range, kRsrcWord3);
}

template <typename T>
__device__ inline T bload(Rsrc r, uint32_t off)
{
    if constexpr (sizeof(T) == 4) {
        return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0));
    } else {
        return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0));
    }
}

template <typename T>
__device__ inline void bstore(T v, Rsrc r, uint32_t off)
{
    if constexpr (sizeof(T) == 4) {
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, v), r, (int)off, 0, 0);
    } else {
        typedef int v2i __attribute__((ext_vector_type(2)));
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2i, v), r, (int)off, 0, 0);
    }
}

}  // namespace scafes
