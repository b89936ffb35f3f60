// Raw buffer addressing for the gfx950 kernels: the base address sits in a 128-bit resource in scalar registers and
// every access takes a 32-bit byte offset per lane plus a scalar offset, so the accesses of a thread share one
// address VGPR and cost no vector address arithmetic. Accesses at or past num_records bytes from the base are not
// performed (loads return 0). Offsets must stay below 4 GiB from the base.
#pragma once

#include "dft.hpp"

namespace crdfft::dev
{

typedef float f2v __attribute__((ext_vector_type(2)));

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t num_records = 0xFFFFFFFFu)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, static_cast<int>(num_records), 0x00020000);
}

// The builtins' own 8-byte vector type (a generic vector, converted as a whole: its elements are not accessed).
using b64_t = decltype(__builtin_amdgcn_raw_buffer_load_b64(make_rsrc(nullptr), 0, 0, 0));
static_assert(sizeof(b64_t) == 8, "64-bit buffer access");
constexpr int kAuxNt = 2; // cache policy of the buffer instructions: non-temporal

template <int AUX> __device__ __forceinline__ cf bld(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff)
{
    const b64_t u = __builtin_amdgcn_raw_buffer_load_b64(r, static_cast<int>(voff), static_cast<int>(soff), AUX);
    const f2v f = __builtin_bit_cast(f2v, u);
    return cf{f.x, f.y};
}

template <int AUX> __device__ __forceinline__ float bld32(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff)
{
    const auto u = __builtin_amdgcn_raw_buffer_load_b32(r, static_cast<int>(voff), static_cast<int>(soff), AUX);
    static_assert(sizeof(u) == 4, "32-bit buffer access");
    return __builtin_bit_cast(float, u);
}

typedef float f4v __attribute__((ext_vector_type(4)));

template <int AUX> __device__ __forceinline__ f4v bld128(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff)
{
    const auto u = __builtin_amdgcn_raw_buffer_load_b128(r, static_cast<int>(voff), static_cast<int>(soff), AUX);
    static_assert(sizeof(u) == 16, "128-bit buffer access");
    return __builtin_bit_cast(f4v, u);
}

template <int AUX> __device__ __forceinline__ void bst32(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff, float v)
{
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r, static_cast<int>(voff),
                                          static_cast<int>(soff), AUX);
}

template <int AUX> __device__ __forceinline__ void bst128(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff, f4v v)
{
    using u4 = decltype(__builtin_amdgcn_raw_buffer_load_b128(r, 0, 0, 0));
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, v), r, static_cast<int>(voff), static_cast<int>(soff),
                                           AUX);
}

template <int AUX> __device__ __forceinline__ void bst(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff, cf v)
{
    f2v f;
    f.x = v.x;
    f.y = v.y;
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(b64_t, f), r, static_cast<int>(voff),
                                          static_cast<int>(soff), AUX);
}

// Which of the sequences of a workgroup (T threads each) a thread belongs to. From T = 64 on the lanes of a wave share
// it, and saying so (readfirstlane) keeps every address that depends on it in scalar registers. Without it a buffer
// resource of the sequence counts as divergent and the compiler makes every access a loop over the resources in the wave
// (11 instructions an iteration), also where there is only one; below T = 64 such loops really run several times, so there
// Row takes plain accesses. Measured on 2^25-point (real: 2^26-sample) batches: DCT-II n = 8 882 -> 92 us, n = 128 61 -> 47;
// chirp-z n = 17 (2^23 points) 173 -> 77, n = 61 81 -> 58; STFT of 2^24 samples, frames of 16 / 64 522 -> 97 / 98 -> 49.
template <int T> __device__ __forceinline__ int slot_of(int tid)
{
    if constexpr (T >= 64)
    {
        return __builtin_amdgcn_readfirstlane(tid / T);
    }
    else
    {
        return tid / T;
    }
}

// One sequence of `bytes` bytes at `base` (0: an inactive slot, base then any sequence of the call). Offsets in bytes,
// voff per lane, soff the same in every lane; elements need 4-byte alignment only.
//   UNIFORM  the same sequence in every lane of a wave: a buffer resource. Loads outside the range return 0, stores
//            outside are dropped.
//   else     several sequences per wave: plain accesses. Stores of inactive slots are dropped, their loads read what is
//            at base; with CHECK every access is held against the range as above.
template <bool UNIFORM, bool CHECK = false> struct Row;

template <bool CHECK> struct Row<true, CHECK>
{
    __amdgpu_buffer_rsrc_t r;
    __device__ __forceinline__ Row(const void* base, uint32_t bytes) : r(make_rsrc(base, bytes)) {}
    __device__ __forceinline__ float ld32(uint32_t voff, uint32_t soff) const { return bld32<0>(r, voff, soff); }
    __device__ __forceinline__ cf ld64(uint32_t voff, uint32_t soff) const { return bld<0>(r, voff, soff); }
    __device__ __forceinline__ f4v ld128(uint32_t voff, uint32_t soff) const { return bld128<0>(r, voff, soff); }
    __device__ __forceinline__ void st32(uint32_t voff, uint32_t soff, float v) const { bst32<0>(r, voff, soff, v); }
    __device__ __forceinline__ void st64(uint32_t voff, uint32_t soff, cf v) const { bst<0>(r, voff, soff, v); }
    __device__ __forceinline__ void st128(uint32_t voff, uint32_t soff, f4v v) const { bst128<0>(r, voff, soff, v); }
};

template <bool CHECK> struct Row<false, CHECK>
{
    typedef float f2u __attribute__((ext_vector_type(2), aligned(4)));
    typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
    const char* p;
    uint32_t n;
    __device__ __forceinline__ Row(const void* base, uint32_t bytes) : p(static_cast<const char*>(base)), n(bytes) {}
    template <class V> __device__ __forceinline__ V get(uint32_t off) const
    {
        if constexpr (CHECK)
        {
            return off < n ? *reinterpret_cast<const V*>(p + off) : V{};
        }
        else
        {
            return *reinterpret_cast<const V*>(p + off);
        }
    }
    template <class V> __device__ __forceinline__ void put(uint32_t off, V v) const
    {
        if (CHECK ? off < n : n != 0)
        {
            *reinterpret_cast<V*>(const_cast<char*>(p) + off) = v;
        }
    }
    __device__ __forceinline__ float ld32(uint32_t voff, uint32_t soff) const { return get<float>(voff + soff); }
    __device__ __forceinline__ cf ld64(uint32_t voff, uint32_t soff) const
    {
        const f2u v = get<f2u>(voff + soff);
        return cf{v.x, v.y};
    }
    __device__ __forceinline__ f4v ld128(uint32_t voff, uint32_t soff) const { return get<f4u>(voff + soff); }
    __device__ __forceinline__ void st32(uint32_t voff, uint32_t soff, float v) const { put<float>(voff + soff, v); }
    __device__ __forceinline__ void st64(uint32_t voff, uint32_t soff, cf v) const
    {
        f2u w;
        w.x = v.x;
        w.y = v.y;
        put<f2u>(voff + soff, w);
    }
    __device__ __forceinline__ void st128(uint32_t voff, uint32_t soff, f4v v) const { put<f4u>(voff + soff, v); }
};

} // namespace crdfft::dev
