// Device-side addressing of the Q8 KV cache and the int8-piece arithmetic its
// MFMA attention kernels share (layout: qwn_attention.hip).
#pragma once

#include "qwn_device.h"

namespace qwn {

// Each KV head's pages are contiguous, so a workgroup streaming one head's
// span of the context reads one contiguous run of keys and one of values.
// key byte of (token, head, channel); channels 16q .. 16q + 15 of a token
// are the 16 bytes at k_index(token, head, 16q)
__device__ __forceinline__ size_t k_index(const KvCache &c, uint32_t token, uint32_t head, uint32_t dim) {
    const uint32_t page = token / kKvPageTokens, slot = token % kKvPageTokens;
    const uint32_t chunks = (c.head_dim + 15) / 16;
    return (((static_cast<size_t>(head) * c.pages + page) * chunks + dim / 16) * kKvPageTokens + slot) * 16 +
           dim % 16;
}

// value byte of (token, head, channel)
__device__ __forceinline__ size_t v_offset(const KvCache &c, uint32_t token, uint32_t head, uint32_t dim) {
    const uint32_t page = token / kKvPageTokens, slot = token % kKvPageTokens;
    return ((static_cast<size_t>(head) * c.pages + page) * c.head_dim + dim) * kKvPageTokens + slot;
}

// the 16 value bytes of (page, head, channel)
__device__ __forceinline__ size_t v_page_offset(const KvCache &c, uint32_t page, uint32_t head, uint32_t dim) {
    return ((static_cast<size_t>(head) * c.pages + page) * c.head_dim + dim) * kKvPageTokens;
}

// scale of (token, group): [group][64-token quad][slot 0..15][page of the
// quad 0..3], so the four floats at scale_index(64q + slot, g) are the
// scales of tokens slot, 16 + slot, 32 + slot, 48 + slot of quad q
__device__ __forceinline__ size_t scale_index(const KvCache &c, uint32_t token, uint32_t group) {
    return ((static_cast<size_t>(group) * c.quads + token / (4 * kKvPageTokens)) * kKvPageTokens +
            token % kKvPageTokens) * 4 + (token / kKvPageTokens) % 4;
}

// Whether slot t is attended under a tree mask relative to slot `base`
// (no tree: a base past every slot).  The 64-bit test is a lookup of
// the mask's two halves by the slot's offset, written without any shift by
// a wrapped offset: an earlier form, t < base || (mask >> min(t - base,
// 63)) & 1, was compiled into the shift alone (the t < base test dropped),
// which masked every token.
__device__ __forceinline__ bool tree_attends(uint32_t t, uint32_t base, uint64_t mask) {
    const uint32_t off = t - base;  // the slot's tree index when t >= base
    const uint32_t half = off < 32u ? static_cast<uint32_t>(mask) : static_cast<uint32_t>(mask >> 32);
    const bool bit = ((half >> (off & 31u)) & 1u) != 0u;
    return t < base || (off < 64u && bit);
}

typedef int att_v4i __attribute__((ext_vector_type(4)));

// Reductions over each 16-lane row by DPP row rotations (row_ror 8, 4, 2,
// 1): every lane of the row ends with the row's max / sum (the sum's
// association differs between lanes; callers read one lane).
template <int CTRL>
__device__ __forceinline__ float dpp_rot(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false));
}
__device__ __forceinline__ float row16_max(float v) {
    v = fmaxf(v, dpp_rot<0x128>(v));
    v = fmaxf(v, dpp_rot<0x124>(v));
    v = fmaxf(v, dpp_rot<0x122>(v));
    return fmaxf(v, dpp_rot<0x121>(v));
}
__device__ __forceinline__ float row16_sum(float v) {
    v += dpp_rot<0x128>(v);
    v += dpp_rot<0x124>(v);
    v += dpp_rot<0x122>(v);
    return v + dpp_rot<0x121>(v);
}

__device__ __forceinline__ float f4_at(const float4 &v, int i) {
    return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w;
}

__device__ __forceinline__ void lds_wave_sync() {
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

}  // namespace qwn
