// Fixed-bit quantisation of a 256-element chunk by one wave, in registers: what the builders and the few-rows linear
// kernel share.
//
// Lane l holds the four consecutive elements chunk_quad(l) .. + 3 of the chunk.  A wave's load of a chunk is then one
// contiguous run (1 KiB of float32), and the permutation of the quads over the lanes puts the four bytes of a dword of the int8
// image (element 32w + 8m + t at byte 32w + 4t + m) into four neighbouring lanes: a 4 x 4 byte transpose inside a quad
// of lanes, two DPP exchanges, leaves lane l with dword l of the image.  From there the planes are an 8 x 8 bit
// transpose over eight neighbouring lanes, three more exchanges.
#pragma once
#include "bsi_dot_device.h"

#include <type_traits>

namespace bsi {

// Chunks whose largest |x| is below 2^16 (as float bits, so that infinities and NaNs are above) are quantised in float32
// arithmetic: with 10^dec <= 127 every magnitude is below 2^23.  The others take the 64-bit routine.
constexpr unsigned kQuantWideBits = 0x47800000u;

__device__ __forceinline__ int chunk_quad(int lane) { return (lane >> 3) * 32 + (lane & 3) * 8 + ((lane >> 2) & 1) * 4; }

struct ChunkLane {
    int quad;                  // first of the lane's four elements
    uint32_t byte1, byte2;     // v_perm selectors of the byte transpose
    uint32_t rot4, rot2, rot1, keep4, keep2, keep1;  // rotations and own-bit masks of the bit transpose
};
__device__ __forceinline__ ChunkLane chunk_lane(int lane) {
    ChunkLane c;
    c.quad = chunk_quad(lane);
    c.byte1 = (lane & 1) ? 0x03070105u : 0x06020400u;
    c.byte2 = (lane & 2) ? 0x03020706u : 0x05040100u;
    c.rot4 = (lane & 4) ? 4u : 28u;
    c.rot2 = (lane & 2) ? 2u : 30u;
    c.rot1 = (lane & 1) ? 1u : 31u;
    c.keep4 = (lane & 4) ? 0xF0F0F0F0u : 0x0F0F0F0Fu;
    c.keep2 = (lane & 2) ? 0xCCCCCCCCu : 0x33333333u;
    c.keep1 = (lane & 1) ? 0xAAAAAAAAu : 0x55555555u;
    return c;
}

template <int kCtrl>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
    return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), kCtrl, 0xF, 0xF, false));
}

// The bytes of the lane's four elements -> the lane's dword of the int8 image.
__device__ __forceinline__ uint32_t chunk_image_dword(uint32_t quad_bytes, const ChunkLane& c) {
    uint32_t v = quad_bytes;
    v = __builtin_amdgcn_perm(dpp_u32<0xB1>(v), v, c.byte1);  // quad_perm [1, 0, 3, 2]
    v = __builtin_amdgcn_perm(dpp_u32<0x4E>(v), v, c.byte2);  // quad_perm [2, 3, 0, 1]
    return v;
}

// The lane's dword of the image -> 32 bits of one plane: image bit b = lane % 8 of elements 32 (lane / 8) .. + 31.
__device__ __forceinline__ uint32_t chunk_plane_dword(uint32_t image, const ChunkLane& c) {
    uint32_t v = image;
    uint32_t o = dpp_u32<0x1B>(dpp_u32<0x141>(v));  // lane ^ 7 (row_half_mirror), then lane ^ 3: lane ^ 4
    v = bsel(v, __builtin_amdgcn_alignbit(o, o, c.rot4), c.keep4);
    o = dpp_u32<0x4E>(v);
    v = bsel(v, __builtin_amdgcn_alignbit(o, o, c.rot2), c.keep2);
    o = dpp_u32<0xB1>(v);
    return bsel(v, __builtin_amdgcn_alignbit(o, o, c.rot1), c.keep1);
}

// Element i of a buffer of T as float; 0 past the descriptor's range.
template <typename T>
__device__ __forceinline__ float buffer_load_as_float(bsi_rsrc r, int i);
template <>
__device__ __forceinline__ float buffer_load_as_float<float>(bsi_rsrc r, int i) {
    return __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, i * 4, 0, 0));
}
template <>
__device__ __forceinline__ float buffer_load_as_float<__half>(bsi_rsrc r, int i) {
    const unsigned short h = static_cast<unsigned short>(__builtin_amdgcn_raw_buffer_load_b16(r, i * 2, 0, 0));
    return __half2float(__ushort_as_half(h));
}
template <>
__device__ __forceinline__ float buffer_load_as_float<__hip_bfloat16>(bsi_rsrc r, int i) {
    const unsigned short h = static_cast<unsigned short>(__builtin_amdgcn_raw_buffer_load_b16(r, i * 2, 0, 0));
    return __uint_as_float(static_cast<uint32_t>(h) << 16);
}

// Four consecutive elements from element i on: one 16- or 8-byte load (i a multiple of 4, the buffer a multiple of 4
// elements long and aligned to the load's size).  kOnce: a nontemporal load, of what is read once.
template <typename T, bool kOnce>
__device__ __forceinline__ void buffer_load_quad(bsi_rsrc r, int i, float (&v)[4]) {
    constexpr int kCache = kOnce ? 2 : 0;
    if constexpr (std::is_same_v<T, float>) {
        typedef unsigned v4u __attribute__((ext_vector_type(4)));
        const v4u u = __builtin_amdgcn_raw_buffer_load_b128(r, i * 4, 0, kCache);
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = __uint_as_float(u[k]);
    } else {
        typedef unsigned v2u __attribute__((ext_vector_type(2)));
        const v2u u = __builtin_amdgcn_raw_buffer_load_b64(r, i * 2, 0, kCache);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if constexpr (std::is_same_v<T, __half>) v[k] = __half2float(__ushort_as_half(static_cast<unsigned short>(u[k >> 1] >> (16 * (k & 1)))));
            else v[k] = __uint_as_float((k & 1) ? (u[k >> 1] & 0xFFFF0000u) : (u[k >> 1] << 16));
        }
    }
}

// The lane's four elements of chunk c of a row; 0 past the row's end.  kVec: d and the row's address allow buffer_load_quad.
template <typename T, bool kVec, bool kOnce = false>
__device__ __forceinline__ void load_chunk_quad(const T* row, int64_t d, int c, const ChunkLane& cl, float (&v)[4]) {
    const bsi_rsrc r = make_rsrc(row, static_cast<size_t>(d) * sizeof(T));
    const int i = c * BSI_CHUNK_ELEMS + cl.quad;
    if (kVec) {
        buffer_load_quad<T, kOnce>(r, i, v);
    } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = buffer_load_as_float<T>(r, i + k);
    }
}

__device__ __forceinline__ unsigned quad_max_bits(const float (&v)[4]) {
    unsigned m = 0u;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const unsigned b = __float_as_uint(v[k]) & 0x7fffffffu;
        m = b > m ? b : m;
    }
    return m;
}

// floor(a * scale + 0.5) as a float, for 0 <= a < 2^16 and an integer scale of at most 127: the integer the exact
// product rounded half away from zero gives.  Half types: a has at most 11 significant bits, so the product is exact
// in float32 and adding 0.5 rounds only where the sum is below 1 anyway.  float32: the fused multiply-add may round
// up to an integer that the exact value does not reach; the sign of a second one, exact where it matters, tells.
template <typename T>
__device__ __forceinline__ float scaled_magnitude_f32(float a, float scale) {
    return truncf(fmaf(a, scale, 0.5f));
}
template <>
__device__ __forceinline__ float scaled_magnitude_f32<float>(float a, float scale) {
    const float t = truncf(fmaf(a, scale, 0.5f));
    return fmaf(a, scale, 0.5f - t) < 0.0f ? t - 1.0f : t;
}

// Shift of a chunk (or row) whose largest |x| has the float bits mx: compute_shift without clipping.
__device__ __forceinline__ int quant_shift(unsigned mx, float scale, int slices) {
    const float t = scaled_magnitude_f32<float>(__uint_as_float(mx), scale);
    const int shift = static_cast<int>(__float_as_uint(t) >> 23) - 126 - (slices - 1);  // bits of t, negative for t = 0
    return shift < 0 ? 0 : shift;
}

struct QuantRange {
    float lo, hi, up;  // the clamp's ends and 2^(8 - slices), which puts the sign bit on the byte's top bit
};
__device__ __forceinline__ QuantRange quant_range(int slices) {
    QuantRange r;
    r.hi = static_cast<float>((1 << (slices - 1)) - 1);
    r.lo = -r.hi - 1.0f;
    r.up = static_cast<float>(1 << (8 - slices));
    return r;
}

__device__ __forceinline__ uint32_t pack_low_bytes(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    return __builtin_amdgcn_perm(__builtin_amdgcn_perm(d, c, 0x0c0c0400u), __builtin_amdgcn_perm(b, a, 0x0c0c0400u), 0x05040100u);
}

// Four elements (|v| < 2^16) rounded, shifted with rounding, clamped and put into the bytes of a dword, each shifted up
// to the byte's top.  Every step is exact: magnitudes are integers below 2^23, dividing by 2^shift and adding 0.5
// leaves at most 24 significant bits, and adding 1.5 * 2^23 leaves the two's complement byte in the low mantissa bits.
template <typename T>
__device__ __forceinline__ uint32_t quantise_quad(const float (&v)[4], float scale, int shift, const QuantRange& r) {
    const float inv = __uint_as_float(static_cast<uint32_t>(127 - shift) << 23);
    uint32_t b[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float q = truncf(fmaf(scaled_magnitude_f32<T>(fabsf(v[k]), scale), inv, 0.5f));
        const float s = __builtin_amdgcn_fmed3f(copysignf(q, v[k]), r.lo, r.hi);
        b[k] = __float_as_uint(fmaf(s, r.up, 12582912.0f));
    }
    return pack_low_bytes(b[0], b[1], b[2], b[3]);
}

// The same for any values, in 64-bit integers (rare: kept in rolled form).
__device__ __forceinline__ uint32_t quantise_quad_wide(const float (&v)[4], double dec_scale, int shift, int slices) {
    const long long qmax = (1LL << (slices - 1)) - 1LL, qmin = -(1LL << (slices - 1));
    uint32_t out = 0u;
#pragma unroll 1
    for (int k = 0; k < 4; ++k) {
        const float x = k == 0 ? v[0] : (k == 1 ? v[1] : (k == 2 ? v[2] : v[3]));
        const long long q = shift_clamp(round_scaled(x, dec_scale), shift, qmin, qmax);
        out |= static_cast<uint32_t>(static_cast<uint8_t>(static_cast<int>(q) << (8 - slices))) << (8 * k);
    }
    return out;
}
__device__ __forceinline__ unsigned long long quad_max_wide(const float (&v)[4], double dec_scale) {
    unsigned long long m = 0ULL;
#pragma unroll 1
    for (int k = 0; k < 4; ++k) {
        const float x = k == 0 ? v[0] : (k == 1 ? v[1] : (k == 2 ? v[2] : v[3]));
        const unsigned long long a = uabs_ll(round_scaled(x, dec_scale));
        m = a > m ? a : m;
    }
    return m;
}

}  // namespace bsi
