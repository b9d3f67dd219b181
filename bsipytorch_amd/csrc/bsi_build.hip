// BSI builder for gfx950: float -> rounded decimal ints -> block-floating shift -> fixed-bit
// two's-complement values -> bit-planes in canonical [rows, slices, W64] words.
//
// wave64 mapping of the general kernels: one wavefront owns one 256-element chunk of one row.  A lane
// loads elements lane, lane+64, lane+128, lane+192 of the chunk (four fully coalesced 256-byte wave
// loads), the chunk maximum is a butterfly reduction across the wave, and one 64-bit `__ballot` per
// slice per load IS the packed plane word (no lo/hi merge, no LDS, no block barrier).  The chunk-scale
// build is therefore a single pass over the activations.  The *_fast kernels (at most 8 slices, 0 to 2
// decimal places, no clipping) hold four consecutive elements a lane instead (bsi_quant_device.h).
//
// Arithmetic follows the reference's quantiser kernels (bsi_ops/csrc/cuda/bsi_cuda_kernels_quant.cuh:
// rounding :24-29, shift :82-108, rounded shift + clamp :205-226) and packer
// (bsi_cuda_kernels_pack.cuh:129-174).
#include "bsi_quant_device.h"

#include <type_traits>

namespace bsi {

constexpr int kBlock = 256;
constexpr int kWavesPerBlock = kBlock / BSI_WAVE;

// ---------------------------------------------------------------- elementwise

template <typename T>
__global__ void round_to_int64_kernel(const T* __restrict__ x, int64_t total, double dec_scale,
                                      long long* __restrict__ out) {
    const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < total; i += stride)
        out[i] = round_scaled(load_as_float<T>(x, i), dec_scale);
}

// (long long)(x * factor) with the product rounded to float first and the conversion towards zero: the scalar
// entry points' value rule (bsiFunctions.cpp:265-271)
template <typename T>
__global__ void trunc_to_int64_kernel(const T* __restrict__ x, int64_t total, float factor, long long* __restrict__ out) {
    const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < total; i += stride)
        out[i] = static_cast<long long>(__fmul_rn(load_as_float<T>(x, i), factor));
}

__global__ void apply_shift_clamp_kernel(long long* __restrict__ ints, int64_t total, int64_t d, int chunks,
                                         const int* __restrict__ shifts, long long qmin, long long qmax) {
    // chunks == 0: one shift per row; else one per (row, col >> 8)
    const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < total; i += stride) {
        const int64_t row = i / d;
        int shift;
        if (chunks > 0) {
            int c = static_cast<int>((i - row * d) >> 8);
            if (c >= chunks) c = chunks - 1;
            shift = shifts[row * chunks + c];
        } else {
            shift = shifts[row];
        }
        ints[i] = shift_clamp(ints[i], shift, qmin, qmax);
    }
}

// ---------------------------------------------------------------- shift / scale passes

// Source of rounded ints: either the float input (rounded on the fly) or staged int64.
template <typename T>
struct RoundedFromInput {
    const T* x;
    double dec_scale;
    __device__ __forceinline__ long long operator()(int64_t i) const { return round_scaled(load_as_float<T>(x, i), dec_scale); }
};
struct RoundedFromInts {
    const long long* v;
    __device__ __forceinline__ long long operator()(int64_t i) const { return v[i]; }
};

// One wave per (row, chunk).
template <typename Src>
__global__ void chunk_shift_scale_kernel(Src src, int64_t Q, int64_t d, int chunks, int fixed_bits, float clip_k,
                                         int* __restrict__ shifts, float* __restrict__ scales) {
    const int lane = threadIdx.x & (BSI_WAVE - 1);
    const int64_t wave = static_cast<int64_t>(blockIdx.x) * kWavesPerBlock + (threadIdx.x >> 6);
    if (wave >= Q * chunks) return;
    const int64_t row = wave / chunks;
    const int c = static_cast<int>(wave - row * chunks);
    const int64_t start = static_cast<int64_t>(c) * BSI_CHUNK_ELEMS;
    int64_t valid = d - start;
    if (valid > BSI_CHUNK_ELEMS) valid = BSI_CHUNK_ELEMS;
    if (valid < 0) valid = 0;
    unsigned long long mx = 0ULL;
    double sum = 0.0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int e = k * BSI_WAVE + lane;
        if (e < valid) {
            const unsigned long long av = uabs_ll(src(row * d + start + e));
            if (av > mx) mx = av;
            sum += static_cast<double>(av);
        }
    }
    mx = wave_max_u64(mx);
    sum = wave_sum_f64(sum);
    if (lane == 0) {
        const int shift = (valid > 0) ? compute_shift(mx, sum, static_cast<int>(valid), fixed_bits, clip_k) : 0;
        shifts[wave] = shift;
        scales[wave] = static_cast<float>(1ULL << shift);
    }
}

// One block per row.
template <typename Src>
__global__ void row_shift_scale_kernel(Src src, int64_t Q, int64_t d, int fixed_bits, float clip_k,
                                       int* __restrict__ shifts, float* __restrict__ scales) {
    __shared__ unsigned long long smax[kWavesPerBlock];
    __shared__ double ssum[kWavesPerBlock];
    const int64_t row = blockIdx.x;
    if (row >= Q) return;
    unsigned long long mx = 0ULL;
    double sum = 0.0;
    for (int64_t e = threadIdx.x; e < d; e += kBlock) {
        const unsigned long long av = uabs_ll(src(row * d + e));
        if (av > mx) mx = av;
        sum += static_cast<double>(av);
    }
    mx = wave_max_u64(mx);
    sum = wave_sum_f64(sum);
    if ((threadIdx.x & (BSI_WAVE - 1)) == 0) {
        smax[threadIdx.x >> 6] = mx;
        ssum[threadIdx.x >> 6] = sum;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kWavesPerBlock; ++w) {
            if (smax[w] > mx) mx = smax[w];
            sum += ssum[w];
        }
        const int shift = compute_shift(mx, sum, static_cast<int>(d), fixed_bits, clip_k);
        shifts[row] = shift;
        scales[row] = static_cast<float>(1ULL << shift);
    }
}

// ---------------------------------------------------------------- pack

// Ballot-pack the four 64-element groups of one chunk held as v[0..3] (low `slices` bits valid) and
// store words 4c..4c+3 of every slice.  Lane s keeps slice s, so each active lane issues one
// contiguous run of stores.
__device__ __forceinline__ void ballot_pack_store(const unsigned long long v[4], int slices, int lane, int c,
                                                  int words_per_slice, unsigned long long* __restrict__ out_row) {
    unsigned long long keep[4] = {0ULL, 0ULL, 0ULL, 0ULL};
    for (int s = 0; s < slices; ++s) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const unsigned long long word = __ballot(((v[k] >> s) & 1ULL) != 0ULL);
            if (lane == (s & (BSI_WAVE - 1))) keep[k] = word;
        }
        if (lane == (s & (BSI_WAVE - 1))) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int w = c * BSI_CHUNK_WORDS + k;
                if (w < words_per_slice) out_row[static_cast<size_t>(s) * words_per_slice + w] = keep[k];
            }
        }
    }
}

// Quantise (given shifts) + pack.  chunks > 0: shift per (row, chunk); chunks == 0: shift per row.
// One wave per (row, group of 4 words).
template <typename Src, bool kQuantise>
__global__ void shift_pack_kernel(Src src, int64_t Q, int64_t d, int chunks, int slices, int words_per_slice,
                                  int fixed_bits, const int* __restrict__ shifts, unsigned long long* __restrict__ out) {
    const int lane = threadIdx.x & (BSI_WAVE - 1);
    const int groups = (words_per_slice + BSI_CHUNK_WORDS - 1) / BSI_CHUNK_WORDS;
    const int64_t wave = static_cast<int64_t>(blockIdx.x) * kWavesPerBlock + (threadIdx.x >> 6);
    if (wave >= Q * groups) return;
    const int64_t row = wave / groups;
    const int c = static_cast<int>(wave - row * groups);
    const unsigned long long mask = (slices >= 64) ? ~0ULL : ((1ULL << slices) - 1ULL);
    int shift = 0;
    long long qmin = 0, qmax = 0;
    if (kQuantise) {
        int sc = c;
        if (chunks > 0 && sc >= chunks) sc = chunks - 1;
        shift = (chunks > 0) ? shifts[row * chunks + sc] : shifts[row];
        qmax = (1LL << (fixed_bits - 1)) - 1LL;
        qmin = -(1LL << (fixed_bits - 1));
    }
    unsigned long long v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int64_t e = static_cast<int64_t>(c) * BSI_CHUNK_ELEMS + k * BSI_WAVE + lane;
        v[k] = 0ULL;
        if (e < d) {
            long long r = src(row * d + e);
            if (kQuantise) r = shift_clamp(r, shift, qmin, qmax);
            v[k] = static_cast<unsigned long long>(r) & mask;
        }
    }
    ballot_pack_store(v, slices, lane, c, words_per_slice,
                      out + static_cast<size_t>(row) * slices * words_per_slice);
}

// ---------------------------------------------------------------- fused builds

// Chunk-scale build of one (row, chunk) item by one wave: round, reduce, shift, clamp, pack (64-bit
// arithmetic throughout: any magnitude, any slice count, optional clipping).
template <typename T>
__device__ __forceinline__ void build_chunk_item(const T* __restrict__ x, int64_t item, int64_t d, int chunks, int slices,
                                                 int words_per_slice, double dec_scale, float clip_k,
                                                 unsigned long long* __restrict__ words, int* __restrict__ shifts,
                                                 float* __restrict__ scales, int8_t* __restrict__ ints8, int lane) {
    const int64_t row = item / chunks;
    const int c = static_cast<int>(item - row * chunks);
    const int64_t start = static_cast<int64_t>(c) * BSI_CHUNK_ELEMS;
    int64_t valid = d - start;
    if (valid > BSI_CHUNK_ELEMS) valid = BSI_CHUNK_ELEMS;
    if (valid < 0) valid = 0;

    long long r[4];
    unsigned long long mx = 0ULL;
    double sum = 0.0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int e = k * BSI_WAVE + lane;
        r[k] = 0;
        if (e < valid) {
            r[k] = round_scaled(load_as_float<T>(x, row * d + start + e), dec_scale);
            const unsigned long long av = uabs_ll(r[k]);
            if (av > mx) mx = av;
            sum += static_cast<double>(av);
        }
    }
    mx = wave_max_u64(mx);
    if (clip_k > 0.0f) sum = wave_sum_f64(sum);
    const int shift = (valid > 0) ? compute_shift(mx, sum, static_cast<int>(valid), slices, clip_k) : 0;
    if (lane == 0) {
        shifts[item] = shift;
        scales[item] = static_cast<float>(1ULL << shift);
    }
    const long long qmax = (1LL << (slices - 1)) - 1LL;
    const long long qmin = -(1LL << (slices - 1));
    const unsigned long long mask = (1ULL << slices) - 1ULL;
    unsigned long long v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int e = k * BSI_WAVE + lane;
        const long long q = (e < valid) ? shift_clamp(r[k], shift, qmin, qmax) : 0;
        v[k] = static_cast<unsigned long long>(q) & mask;
        if (ints8 != nullptr)
            ints8[static_cast<size_t>(item) * BSI_CHUNK_ELEMS + mfma_byte_pos(e)] =
                static_cast<int8_t>(static_cast<int>(q) << (8 - slices));
    }
    ballot_pack_store(v, slices, lane, c, words_per_slice,
                      words + static_cast<size_t>(row) * slices * words_per_slice);
}

template <typename T>
__global__ void build_fixed_chunk_kernel(const T* __restrict__ x, int64_t Q, int64_t d, int chunks, int slices,
                                         int words_per_slice, double dec_scale, float clip_k,
                                         unsigned long long* __restrict__ words, int* __restrict__ shifts,
                                         float* __restrict__ scales, int8_t* __restrict__ ints8) {
    const int lane = threadIdx.x & (BSI_WAVE - 1);
    const int64_t wave = static_cast<int64_t>(blockIdx.x) * kWavesPerBlock + (threadIdx.x >> 6);
    if (wave >= Q * chunks) return;
    build_chunk_item<T>(x, wave, d, chunks, slices, words_per_slice, dec_scale, clip_k, words, shifts, scales, ints8, lane);
}

// The same build for the common case (at most 8 slices, no clipping, whole chunks of words, 10^dec an integer of at
// most 127): a wave takes kItems consecutive (row, chunk) items, all loads first, and quantises each in registers
// (bsi_quant_device.h).  The lane that loads four consecutive elements is chosen so that two DPP exchanges leave every
// lane with one dword of the int8 image, and three more with one 32-element half-word of one plane: no LDS, and the
// image is written 256 contiguous bytes an item.  kPlanes = false leaves the planes out (a linear layer's dot on the
// matrix cores reads the image only).  Bound by VALU issue at about 90 instructions an item (float32; 70 for half
// types), near the memory time of the larger inputs.
// 4096 x 4096 bfloat16: 47 us through LDS bytes and 32-bit integers, 15.5 us this way, 12.6 us without the planes (50 MB
// at 4 TB/s).
template <typename T, int kItems, bool kVec, bool kPlanes>
__global__ __launch_bounds__(kBlock) void build_fixed_chunk_fast_kernel(
    const T* __restrict__ x, unsigned total, int64_t d, unsigned chunks, int slices, int words_per_slice, double dec_scale,
    float scale, unsigned long long* __restrict__ words, int* __restrict__ shifts, float* __restrict__ scales,
    int8_t* __restrict__ ints8) {
    const int lane = threadIdx.x & (BSI_WAVE - 1);
    const unsigned item0 = (blockIdx.x * kWavesPerBlock + static_cast<unsigned>(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6))) * kItems;
    if (item0 >= total) return;
    const ChunkLane cl = chunk_lane(lane);
    const QuantRange range = quant_range(slices);
    float v[kItems][4];
    unsigned row[kItems], col[kItems];
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
        const unsigned item = item0 + j < total ? item0 + j : total - 1;  // a wave past the end repeats the last item
        row[j] = item / chunks;
        col[j] = item - row[j] * chunks;
        load_chunk_quad<T, kVec>(x + static_cast<int64_t>(row[j]) * d, d, static_cast<int>(col[j]), cl, v[j]);
    }
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
        const unsigned item = item0 + j < total ? item0 + j : total - 1;
        const unsigned mx = wave_max_u32(quad_max_bits(v[j]));
        int shift;
        uint32_t image;
        if (mx < kQuantWideBits) {
            shift = quant_shift(mx, scale, slices);
            image = quantise_quad<T>(v[j], scale, shift, range);
        } else {
            shift = compute_shift(wave_max_u64(quad_max_wide(v[j], dec_scale)), 0.0, BSI_CHUNK_ELEMS, slices, 0.0f);
            image = quantise_quad_wide(v[j], dec_scale, shift, slices);
        }
        image = chunk_image_dword(image, cl);
        if (lane == 0) {
            if (shifts != nullptr) shifts[item] = shift;
            scales[item] = static_cast<float>(1ULL << shift);
        }
        if (ints8 != nullptr) reinterpret_cast<uint32_t*>(ints8)[static_cast<size_t>(item) * (BSI_CHUNK_ELEMS / 4) + lane] = image;
        if (kPlanes) {
            const uint32_t plane = chunk_plane_dword(image, cl);  // by all lanes: it exchanges registers between them
            const int sl = (lane & 7) - (8 - slices);
            if (sl >= 0)
                reinterpret_cast<uint32_t*>(words)[(static_cast<size_t>(row[j]) * slices + sl) * (2 * words_per_slice) +
                                                   col[j] * 8 + (lane >> 3)] = plane;
        }
    }
}

// Row-scale build: one block per row; pass 1 reduces the row maximum, pass 2 (row now in cache)
// quantises and packs, one wave per group of 4 words.
template <typename T>
__global__ void build_fixed_row_kernel(const T* __restrict__ x, int64_t Q, int64_t d, int slices,
                                       int words_per_slice, double dec_scale, float clip_k,
                                       unsigned long long* __restrict__ words, int* __restrict__ shifts,
                                       float* __restrict__ scales, int8_t* __restrict__ ints8) {
    __shared__ unsigned long long smax[kWavesPerBlock];
    __shared__ double ssum[kWavesPerBlock];
    __shared__ int sshift;
    const int64_t row = blockIdx.x;
    if (row >= Q) return;
    const int lane = threadIdx.x & (BSI_WAVE - 1);
    const int wid = threadIdx.x >> 6;
    unsigned long long mx = 0ULL;
    double sum = 0.0;
    for (int64_t e = threadIdx.x; e < d; e += kBlock) {
        const unsigned long long av = uabs_ll(round_scaled(load_as_float<T>(x, row * d + e), dec_scale));
        if (av > mx) mx = av;
        sum += static_cast<double>(av);
    }
    mx = wave_max_u64(mx);
    sum = wave_sum_f64(sum);
    if (lane == 0) {
        smax[wid] = mx;
        ssum[wid] = sum;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kWavesPerBlock; ++w) {
            if (smax[w] > mx) mx = smax[w];
            sum += ssum[w];
        }
        const int shift = compute_shift(mx, sum, static_cast<int>(d), slices, clip_k);
        sshift = shift;
        shifts[row] = shift;
        scales[row] = static_cast<float>(1ULL << shift);
    }
    __syncthreads();
    const int shift = sshift;
    const long long qmax = (1LL << (slices - 1)) - 1LL;
    const long long qmin = -(1LL << (slices - 1));
    const unsigned long long mask = (1ULL << slices) - 1ULL;
    const int groups = (words_per_slice + BSI_CHUNK_WORDS - 1) / BSI_CHUNK_WORDS;
    for (int c = wid; c < groups; c += kWavesPerBlock) {
        unsigned long long v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int el = k * BSI_WAVE + lane;
            const int64_t e = static_cast<int64_t>(c) * BSI_CHUNK_ELEMS + el;
            long long q = 0;
            if (e < d) q = shift_clamp(round_scaled(load_as_float<T>(x, row * d + e), dec_scale), shift, qmin, qmax);
            v[k] = static_cast<unsigned long long>(q) & mask;
            if (ints8 != nullptr)
                ints8[(static_cast<size_t>(row) * groups + c) * BSI_CHUNK_ELEMS + mfma_byte_pos(el)] =
                    static_cast<int8_t>(static_cast<int>(q) << (8 - slices));
        }
        ballot_pack_store(v, slices, lane, c, words_per_slice,
                          words + static_cast<size_t>(row) * slices * words_per_slice);
    }
}

// The row-scale build for the same common case, one workgroup per row: the row's quads stay in registers between the
// maximum and the quantiser (kHeld chunks a wave; the rest of a longer row is loaded again).  Query batches whose width
// is not a whole number of chunks come here.  77 rows of 1600: 11.0 us in two passes of 64-bit arithmetic, 4.8 us.
template <typename T, bool kVec, bool kPlanes>
__global__ __launch_bounds__(kBlock) void build_fixed_row_fast_kernel(const T* __restrict__ x, int64_t d, int chunks, int slices,
                                                                      int words_per_slice, double dec_scale, float scale,
                                                                      unsigned long long* __restrict__ words,
                                                                      int* __restrict__ shifts, float* __restrict__ scales,
                                                                      int8_t* __restrict__ ints8) {
    constexpr int kHeld = 4;
    __shared__ unsigned smax[kWavesPerBlock];
    __shared__ unsigned long long smax64[kWavesPerBlock];
    const int lane = threadIdx.x & (BSI_WAVE - 1);
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t row = blockIdx.x;
    const T* xrow = x + row * d;
    const ChunkLane cl = chunk_lane(lane);
    float v[kHeld][4];
    unsigned mx = 0u;
#pragma unroll
    for (int j = 0; j < kHeld; ++j) load_chunk_quad<T, kVec>(xrow, d, wid + j * kWavesPerBlock, cl, v[j]);  // past the row: zeros
#pragma unroll
    for (int j = 0; j < kHeld; ++j) {
        const unsigned m = quad_max_bits(v[j]);
        mx = m > mx ? m : mx;
    }
    for (int c = wid + kHeld * kWavesPerBlock; c < chunks; c += kWavesPerBlock) {
        float t[4];
        load_chunk_quad<T, kVec>(xrow, d, c, cl, t);
        const unsigned m = quad_max_bits(t);
        mx = m > mx ? m : mx;
    }
    mx = wave_max_u32(mx);
    if (lane == 0) smax[wid] = mx;
    __syncthreads();
    mx = 0u;
#pragma unroll
    for (int w = 0; w < kWavesPerBlock; ++w) mx = smax[w] > mx ? smax[w] : mx;
    const bool wide = mx >= kQuantWideBits;
    int shift = quant_shift(mx, scale, slices);
    if (wide) {
        unsigned long long m64 = 0ULL;
        for (int c = wid; c < chunks; c += kWavesPerBlock) {
            float t[4];
            load_chunk_quad<T, kVec>(xrow, d, c, cl, t);
            const unsigned long long m = quad_max_wide(t, dec_scale);
            m64 = m > m64 ? m : m64;
        }
        m64 = wave_max_u64(m64);
        if (lane == 0) smax64[wid] = m64;
        __syncthreads();
        for (int w = 0; w < kWavesPerBlock; ++w) m64 = smax64[w] > m64 ? smax64[w] : m64;
        shift = compute_shift(m64, 0.0, 1, slices, 0.0f);
    }
    if (threadIdx.x == 0) {
        if (shifts != nullptr) shifts[row] = shift;
        scales[row] = static_cast<float>(1ULL << shift);
    }
    const QuantRange range = quant_range(slices);
    auto emit = [&](int c, const float (&t)[4]) {
        const uint32_t image = chunk_image_dword(wide ? quantise_quad_wide(t, dec_scale, shift, slices)
                                                      : quantise_quad<T>(t, scale, shift, range), cl);
        if (ints8 != nullptr)
            reinterpret_cast<uint32_t*>(ints8)[(static_cast<size_t>(row) * chunks + c) * (BSI_CHUNK_ELEMS / 4) + lane] = image;
        if (kPlanes) {
            const int sl = (lane & 7) - (8 - slices), unit = c * 8 + (lane >> 3);
            const uint32_t plane = chunk_plane_dword(image, cl);
            if (sl >= 0 && unit < 2 * words_per_slice)
                reinterpret_cast<uint32_t*>(words)[(static_cast<size_t>(row) * slices + sl) * (2 * words_per_slice) + unit] = plane;
        }
    };
#pragma unroll
    for (int j = 0; j < kHeld; ++j)
        if (wid + j * kWavesPerBlock < chunks) emit(wid + j * kWavesPerBlock, v[j]);
    for (int c = wid + kHeld * kWavesPerBlock; c < chunks; c += kWavesPerBlock) {
        float t[4];
        load_chunk_quad<T, kVec>(xrow, d, c, cl, t);
        emit(c, t);
    }
}

// Bytes of a quad as sign and magnitude (at most 127) -> shifted right with rounding (half away from zero), clamped and
// moved to the byte's top as two's complement, four at a time: every step stays inside its byte.  The row's largest
// magnitude gave the shift, so that a shifted magnitude is 2^(slices - 1) at most, and only a positive one is one too many.
struct QuadShift {
    uint32_t half, keep, xor_top, keep_top;
    int shift, top, up;
};
__device__ __forceinline__ QuadShift quad_shift(int shift, int slices) {
    QuadShift q;
    q.shift = shift & 7;  // magnitudes of at most 127 never take more
    q.half = ((1u << q.shift) >> 1) * 0x01010101u;
    q.keep = (0xFFu >> q.shift) * 0x01010101u;
    q.top = slices - 1;
    q.up = 8 - slices;
    q.xor_top = slices == 8 ? 0x80808080u : 0u;
    q.keep_top = ((0xFFu << q.up) & 0xFFu) * 0x01010101u;
    return q;
}
__device__ __forceinline__ uint32_t shift_quad_bytes(uint32_t sm, const QuadShift& q) {
    const uint32_t neg1 = (sm >> 7) & 0x01010101u;
    uint32_t m = (((sm & 0x7F7F7F7Fu) + q.half) >> q.shift) & q.keep;
    m -= (m >> q.top) & (neg1 ^ 0x01010101u);
    const uint32_t minus = m & ((neg1 << 8) - neg1);
    const uint32_t biased = m + 0x80808080u - (minus << 1);  // 128 + the signed value
    return ((biased << q.up) & q.keep_top) ^ q.xor_top;
}

// The whole of a fixed-bit key build for the common case: one workgroup = 16 rows (a tile of the tiled planes), a wave
// each.  A wave reads its row once: the rounded magnitudes and signs of the first kHeld chunks stay in registers as bytes
// until the row's maximum is known (a row with a magnitude over 127, |x| of 1.27 at two decimal places, and the rest of a
// longer row are read again).  It writes the int8 image, 256 contiguous bytes a chunk, and puts its planes' half-words
// into LDS, from where the workgroup writes the tile's words of eight chunks at a time as one contiguous run (a row's own
// words lie 128 bytes apart there).  Slice weights and shifts come out of the same launch.
//
// Memory and VALU work are of the same order here (16384 x 4096 float32: 387 MB, 75 us at the rate of a large copy), and a
// workgroup alternates between the two, so that two of them share a CU: 64 registers (with one a CU 8192 x 5120 bfloat16
// takes 44 us instead of 31).  Float32 arithmetic rounds towards zero throughout the kernel: a * 10^dec + 0.5 then never rounds up to an integer that the exact
// value does not reach, the conversion to a byte truncates, and every other float operation here is exact.
// The stores are nontemporal: nobody reads the planes or the image before the launch is over, and lines that wait in the
// L2s are written back at its end.  Before (16-bit pairs in registers for up to 16 chunks, plain stores) and now, us:
// 16384 x 4096 float32 94.9 -> 79.2 (4.9 TB/s), 8192 x 8192 119.4 -> 85.7, 4096 x 4096 22.5 -> 18.6, 768 x 768 6.7 -> 4.5;
// bfloat16 16384 x 4096 64.2 -> 54.3, 8192 x 5120 37.4 -> 26.7, 2048 x 2048 8.4 -> 7.3.
// kOnce: the loads are nontemporal too, for matrices that the memory-side cache does not hold, of whole lines (a line that two
// rows share is fetched twice, 12800 x 1000 float32 15.8, 17.9).  us, plain and nontemporal: 16384 x 4096 float32 79.4, 75.7,
// bfloat16 54.3, 52.7; 11008 x 4096 float16 38.9, 36.4; below the line 4096 x 4096 float32 (64 MiB) 21.1, 21.6.
// Rows of 17 to 32 chunks, with four loads of a wave in flight instead of eight, pay more for a miss, and their line lies
// higher: 8192 x 8192 float32 86.7, 78.3, bfloat16 59.9, 54.5; 13000 x 5120 float32 82.8, 78.9; of 108 MB 3295 x 8192 float32
// 36.3, 35.3, 12408 x 4352 bfloat16 48.4, 47.8; of 100 MB 3051 x 8192 float32 34.9, 35.6; of 84 MB 8203 x 5120 bfloat16 32.0, 39.3.
constexpr size_t kKeysOnceBytes = size_t{80} << 20, kKeysOnceLongBytes = size_t{100} << 20;
constexpr int kKeyRows = 16, kKeyGroup = 8;
template <typename T, bool kVec, int kHeld, int kLoads, bool kOnce>
__global__ __launch_bounds__(kKeyRows * BSI_WAVE, 8) void build_keys_fast_kernel(
    const T* __restrict__ x, int64_t R, int64_t d, int chunks, int slices, double dec_scale, float scale,
    unsigned long long* __restrict__ tiled, int8_t* __restrict__ image8, int* __restrict__ shifts, float* __restrict__ weights) {
    // [chunk][slice][word of the chunk][row], rows padded to 17 so that the half-words of a wave spread over the banks
    constexpr int kWordStride = 17, kSliceStride = 4 * kWordStride, kChunkStride = 8 * kSliceStride;
    __shared__ unsigned long long stage[kKeyGroup * kChunkStride];
    __builtin_amdgcn_s_setreg(1 | (1 << 11), 3);  // MODE, the two rounding bits of float32: towards zero
    const int lane = threadIdx.x & (BSI_WAVE - 1);
    const int rr = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t row = static_cast<int64_t>(blockIdx.x) * kKeyRows + rr;
    const bool have = row < R;
    const T* xrow = x + (have ? row : R - 1) * d;
    const ChunkLane cl = chunk_lane(lane);
    uint32_t held[kHeld];
    float mxf = 0.0f;
    auto take_max = [&](const float (&v)[4]) {  // a NaN stays
        mxf = __builtin_elementwise_maximum(__builtin_elementwise_maximum(mxf, fabsf(v[0])), fabsf(v[1]));
        mxf = __builtin_elementwise_maximum(__builtin_elementwise_maximum(mxf, fabsf(v[2])), fabsf(v[3]));
    };
#pragma unroll
    for (int c = 0; c < kHeld; c += kLoads) {
        if (c >= chunks) break;
        float v[kLoads][4];
#pragma unroll
        for (int j = 0; j < kLoads; ++j) load_chunk_quad<T, kVec, kOnce>(xrow, d, c + j, cl, v[j]);  // past the row: zeros
#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
            take_max(v[j]);
            uint32_t m = 0u;
            m = __builtin_amdgcn_cvt_pk_u8_f32(fmaf(fabsf(v[j][0]), scale, 0.5f), 0, m);
            m = __builtin_amdgcn_cvt_pk_u8_f32(fmaf(fabsf(v[j][1]), scale, 0.5f), 1, m);
            m = __builtin_amdgcn_cvt_pk_u8_f32(fmaf(fabsf(v[j][2]), scale, 0.5f), 2, m);
            m = __builtin_amdgcn_cvt_pk_u8_f32(fmaf(fabsf(v[j][3]), scale, 0.5f), 3, m);
            const uint32_t signs = __builtin_amdgcn_perm(
                __builtin_amdgcn_perm(__float_as_uint(v[j][3]), __float_as_uint(v[j][2]), 0x0c0c0703u),
                __builtin_amdgcn_perm(__float_as_uint(v[j][1]), __float_as_uint(v[j][0]), 0x0c0c0703u), 0x05040100u);
            held[c + j] = bsel(m, signs, 0x7F7F7F7Fu);
            asm volatile("" : "+v"(held[c + j]));  // packed here: sunk to its use it would keep four registers instead of one
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    for (int c = kHeld; c < chunks; ++c) {
        float v[4];
        load_chunk_quad<T, kVec>(xrow, d, c, cl, v);
        take_max(v);
    }
    const unsigned mx = __builtin_amdgcn_readfirstlane(wave_max_u32(__float_as_uint(mxf) & 0x7FFFFFFFu));
    const bool wide = mx >= kQuantWideBits;
    const bool in_bytes = !wide && scaled_magnitude_f32<float>(__uint_as_float(mx), scale) <= 127.0f;
    int shift = quant_shift(mx, scale, slices);
    if (wide) {
        unsigned long long m64 = 0ULL;
        for (int c = 0; c < chunks; ++c) {
            float v[4];
            load_chunk_quad<T, kVec>(xrow, d, c, cl, v);
            const unsigned long long m = quad_max_wide(v, dec_scale);
            m64 = m > m64 ? m : m64;
        }
        shift = compute_shift(wave_max_u64(m64), 0.0, 1, slices, 0.0f);
    }
    shift = __builtin_amdgcn_readfirstlane(shift);
    if (have && lane < slices) {
        const float w = static_cast<float>(1ULL << shift) * static_cast<float>(1 << lane);
        weights[row * slices + lane] = lane == slices - 1 ? -w : w;
        if (lane == 0) shifts[row] = shift;
    }
    const QuantRange range = quant_range(slices);
    const QuadShift in_byte = quad_shift(shift, slices);
    auto group = [&](int c0, auto first_held) {
        constexpr int kFirst = decltype(first_held)::value;  // the group's first chunk in `held`, or -1
        const int n = chunks - c0 < kKeyGroup ? chunks - c0 : kKeyGroup;
#pragma unroll
        for (int u = 0; u < kKeyGroup; ++u) {
            const int c = c0 + u;
            if (u < n) {
                uint32_t bytes;
                if (kFirst >= 0 && in_bytes) {
                    bytes = shift_quad_bytes(held[(kFirst < 0 ? 0 : kFirst) + u], in_byte);
                } else {
                    float v[4];
                    load_chunk_quad<T, kVec>(xrow, d, c, cl, v);
                    bytes = wide ? quantise_quad_wide(v, dec_scale, shift, slices) : quantise_quad<T>(v, scale, shift, range);
                }
                const uint32_t image = chunk_image_dword(bytes, cl);
                if (have) __builtin_nontemporal_store(image, reinterpret_cast<uint32_t*>(image8) + (static_cast<size_t>(row) * chunks + c) * (BSI_CHUNK_ELEMS / 4) + lane);
                const int sl = (lane & 7) - (8 - slices), unit = lane >> 3;
                const uint32_t plane = chunk_plane_dword(image, cl);
                if (sl >= 0)
                    reinterpret_cast<uint32_t*>(stage)[(u * kChunkStride + sl * kSliceStride + (unit >> 1) * kWordStride + rr) * 2 + (unit & 1)] =
                        have ? plane : 0u;
            }
        }
        __syncthreads();
        // a chunk's words by 512 threads (there are slices * 64 of them): thread w % 512 = slice * 64 + word * 16 + row
        const int w = threadIdx.x & 511, words = slices * 64;
        unsigned long long* dst = tiled + (static_cast<size_t>(blockIdx.x) * chunks + c0) * words + w;
        const unsigned long long* src = stage + (w >> 6) * kSliceStride + ((w >> 4) & 3) * kWordStride + (w & 15);
        if (w < words) {
#pragma unroll
            for (int u = 0; u < kKeyGroup; u += 2) {
                const int v = u + (rr >> 3);
                if (v < n) __builtin_nontemporal_store(src[v * kChunkStride], dst + static_cast<size_t>(v) * words);
            }
        }
        __syncthreads();
    };
    group(0, std::integral_constant<int, 0>{});
    if (kHeld > 8 && chunks > 8) group(8, std::integral_constant<int, (kHeld > 8) ? 8 : -1>{});
    if (kHeld > 16 && chunks > 16) group(16, std::integral_constant<int, (kHeld > 16) ? 16 : -1>{});
    if (kHeld > 24 && chunks > 24) group(24, std::integral_constant<int, (kHeld > 24) ? 24 : -1>{});
    for (int c0 = kHeld; c0 < chunks; c0 += kKeyGroup) group(c0, std::integral_constant<int, -1>{});
}

static inline unsigned grid_for(int64_t waves) {
    return static_cast<unsigned>((waves + kWavesPerBlock - 1) / kWavesPerBlock);
}
static inline unsigned grid_elementwise(int64_t total) {
    int64_t b = (total + kBlock - 1) / kBlock;
    if (b > 65535 * 16) b = 65535 * 16;
    if (b < 1) b = 1;
    return static_cast<unsigned>(b);
}

}  // namespace bsi

using namespace bsi;

#define BSI_DISPATCH_DTYPE(dtype, ...)                                                   \
    switch (dtype) {                                                                     \
        case BSI_DTYPE_F32: { using T = float; __VA_ARGS__; break; }                     \
        case BSI_DTYPE_F16: { using T = __half; __VA_ARGS__; break; }                    \
        case BSI_DTYPE_BF16: { using T = __hip_bfloat16; __VA_ARGS__; break; }           \
        default: return fail(BSI_ERR_INVALID, "unknown dtype code %d", dtype);           \
    }

extern "C" int bsi_hip_quantize_round_to_int64(const void* x, int dtype, int64_t total, double dec_scale,
                                               int64_t* out, void* stream) {
    BSI_REQUIRE(total >= 0, "total must be >= 0");
    if (total == 0) return BSI_OK;
    BSI_REQUIRE(x && out, "null pointer");
    BSI_DISPATCH_DTYPE(dtype, launch(round_to_int64_kernel<T>, dim3(grid_elementwise(total)), dim3(kBlock),
                                                 0, as_stream(stream), static_cast<const T*>(x), total, dec_scale,
                                                 reinterpret_cast<long long*>(out)));
    BSI_LAUNCH_CHECK("round_to_int64_kernel");
    return BSI_OK;
}

extern "C" int bsi_hip_quantize_trunc_to_int64(const void* x, int dtype, int64_t total, float factor, int64_t* out,
                                               void* stream) {
    BSI_REQUIRE(total >= 0, "total must be >= 0");
    if (total == 0) return BSI_OK;
    BSI_REQUIRE(x && out, "null pointer");
    BSI_DISPATCH_DTYPE(dtype, launch(trunc_to_int64_kernel<T>, dim3(grid_elementwise(total)), dim3(kBlock),
                                                 0, as_stream(stream), static_cast<const T*>(x), total, factor,
                                                 reinterpret_cast<long long*>(out)));
    BSI_LAUNCH_CHECK("trunc_to_int64_kernel");
    return BSI_OK;
}

extern "C" int bsi_hip_compute_row_shift_scale(const int64_t* ints, int64_t Q, int64_t d, int fixed_bits, float clip_k,
                                               int32_t* shifts, float* scales, void* stream) {
    BSI_REQUIRE(Q >= 0 && d >= 0, "negative size");
    if (Q == 0) return BSI_OK;
    BSI_REQUIRE(ints && shifts && scales, "null pointer");
    RoundedFromInts src{reinterpret_cast<const long long*>(ints)};
    launch(row_shift_scale_kernel<RoundedFromInts>, dim3(static_cast<unsigned>(Q)), dim3(kBlock), 0,
                       as_stream(stream), src, Q, d, fixed_bits, clip_k, shifts, scales);
    BSI_LAUNCH_CHECK("row_shift_scale_kernel");
    return BSI_OK;
}

extern "C" int bsi_hip_compute_chunk_shift_scale(const int64_t* ints, int64_t Q, int64_t d, int chunks, int fixed_bits,
                                                 float clip_k, int32_t* shifts, float* scales, void* stream) {
    BSI_REQUIRE(Q >= 0 && d >= 0 && chunks >= 0, "negative size");
    if (Q == 0 || chunks == 0) return BSI_OK;
    BSI_REQUIRE(ints && shifts && scales, "null pointer");
    RoundedFromInts src{reinterpret_cast<const long long*>(ints)};
    launch(chunk_shift_scale_kernel<RoundedFromInts>, dim3(grid_for(Q * chunks)), dim3(kBlock), 0,
                       as_stream(stream), src, Q, d, chunks, fixed_bits, clip_k, shifts, scales);
    BSI_LAUNCH_CHECK("chunk_shift_scale_kernel");
    return BSI_OK;
}

extern "C" int bsi_hip_apply_row_shift_clamp(int64_t* ints, int64_t Q, int64_t d, const int32_t* shifts, int fixed_bits,
                                             void* stream) {
    BSI_REQUIRE(Q >= 0 && d >= 0, "negative size");
    BSI_REQUIRE(fixed_bits >= 2 && fixed_bits <= 63, "fixed_bits must be in [2, 63]");
    if (Q == 0 || d == 0) return BSI_OK;
    BSI_REQUIRE(ints && shifts, "null pointer");
    launch(apply_shift_clamp_kernel, dim3(grid_elementwise(Q * d)), dim3(kBlock), 0, as_stream(stream),
                       reinterpret_cast<long long*>(ints), Q * d, d, 0, shifts, -(1LL << (fixed_bits - 1)),
                       (1LL << (fixed_bits - 1)) - 1LL);
    BSI_LAUNCH_CHECK("apply_shift_clamp_kernel");
    return BSI_OK;
}

extern "C" int bsi_hip_apply_chunk_shift_clamp(int64_t* ints, int64_t Q, int64_t d, int chunks, const int32_t* shifts,
                                               int fixed_bits, void* stream) {
    BSI_REQUIRE(Q >= 0 && d >= 0 && chunks > 0, "bad size");
    BSI_REQUIRE(fixed_bits >= 2 && fixed_bits <= 63, "fixed_bits must be in [2, 63]");
    if (Q == 0 || d == 0) return BSI_OK;
    BSI_REQUIRE(ints && shifts, "null pointer");
    launch(apply_shift_clamp_kernel, dim3(grid_elementwise(Q * d)), dim3(kBlock), 0, as_stream(stream),
                       reinterpret_cast<long long*>(ints), Q * d, d, chunks, shifts, -(1LL << (fixed_bits - 1)),
                       (1LL << (fixed_bits - 1)) - 1LL);
    BSI_LAUNCH_CHECK("apply_shift_clamp_kernel");
    return BSI_OK;
}

extern "C" int bsi_hip_compute_row_shift_scale_from_input(const void* x, int dtype, int64_t Q, int64_t d,
                                                          double dec_scale, int fixed_bits, float clip_k,
                                                          int32_t* shifts, float* scales, void* stream) {
    BSI_REQUIRE(Q >= 0 && d >= 0, "negative size");
    if (Q == 0) return BSI_OK;
    BSI_REQUIRE(x && shifts && scales, "null pointer");
    BSI_DISPATCH_DTYPE(dtype, {
        RoundedFromInput<T> src{static_cast<const T*>(x), dec_scale};
        launch(row_shift_scale_kernel<RoundedFromInput<T>>, dim3(static_cast<unsigned>(Q)), dim3(kBlock),
                           0, as_stream(stream), src, Q, d, fixed_bits, clip_k, shifts, scales);
    });
    BSI_LAUNCH_CHECK("row_shift_scale_kernel");
    return BSI_OK;
}

extern "C" int bsi_hip_compute_chunk_shift_scale_from_input(const void* x, int dtype, int64_t Q, int64_t d, int chunks,
                                                            double dec_scale, int fixed_bits, float clip_k,
                                                            int32_t* shifts, float* scales, void* stream) {
    BSI_REQUIRE(Q >= 0 && d >= 0 && chunks >= 0, "negative size");
    if (Q == 0 || chunks == 0) return BSI_OK;
    BSI_REQUIRE(x && shifts && scales, "null pointer");
    BSI_DISPATCH_DTYPE(dtype, {
        RoundedFromInput<T> src{static_cast<const T*>(x), dec_scale};
        launch(chunk_shift_scale_kernel<RoundedFromInput<T>>, dim3(grid_for(Q * chunks)), dim3(kBlock), 0,
                           as_stream(stream), src, Q, d, chunks, fixed_bits, clip_k, shifts, scales);
    });
    BSI_LAUNCH_CHECK("chunk_shift_scale_kernel");
    return BSI_OK;
}

static int check_pack_args(int64_t Q, int64_t d, int slices, int words_per_slice) {
    BSI_REQUIRE(Q >= 0 && d >= 0, "negative size");
    BSI_REQUIRE(slices >= 1 && slices <= 64, "slices must be in [1, 64]");
    BSI_REQUIRE(words_per_slice >= 1 && static_cast<int64_t>(words_per_slice) * 64 >= d,
                "words_per_slice * 64 must cover d");
    return BSI_OK;
}

extern "C" int bsi_hip_quantize_shift_pack_row_batch(const void* x, int dtype, int64_t Q, int64_t d, int slices,
                                                     int words_per_slice, double dec_scale, int fixed_bits,
                                                     const int32_t* shifts, uint64_t* words, void* stream) {
    if (int rc = check_pack_args(Q, d, slices, words_per_slice)) return rc;
    BSI_REQUIRE(fixed_bits >= 2 && fixed_bits <= 63, "fixed_bits must be in [2, 63]");
    if (Q == 0) return BSI_OK;
    BSI_REQUIRE(x && shifts && words, "null pointer");
    const int groups = (words_per_slice + 3) / 4;
    BSI_DISPATCH_DTYPE(dtype, {
        RoundedFromInput<T> src{static_cast<const T*>(x), dec_scale};
        launch((shift_pack_kernel<RoundedFromInput<T>, true>), dim3(grid_for(Q * groups)), dim3(kBlock), 0,
                           as_stream(stream), src, Q, d, 0, slices, words_per_slice, fixed_bits, shifts,
                           reinterpret_cast<unsigned long long*>(words));
    });
    BSI_LAUNCH_CHECK("shift_pack_kernel");
    return BSI_OK;
}

extern "C" int bsi_hip_quantize_shift_pack_chunk_batch(const void* x, int dtype, int64_t Q, int64_t d, int chunks,
                                                       int slices, int words_per_slice, double dec_scale,
                                                       int fixed_bits, const int32_t* shifts, uint64_t* words,
                                                       void* stream) {
    if (int rc = check_pack_args(Q, d, slices, words_per_slice)) return rc;
    BSI_REQUIRE(fixed_bits >= 2 && fixed_bits <= 63, "fixed_bits must be in [2, 63]");
    BSI_REQUIRE(chunks > 0, "chunks must be > 0");
    if (Q == 0) return BSI_OK;
    BSI_REQUIRE(x && shifts && words, "null pointer");
    const int groups = (words_per_slice + 3) / 4;
    BSI_DISPATCH_DTYPE(dtype, {
        RoundedFromInput<T> src{static_cast<const T*>(x), dec_scale};
        launch((shift_pack_kernel<RoundedFromInput<T>, true>), dim3(grid_for(Q * groups)), dim3(kBlock), 0,
                           as_stream(stream), src, Q, d, chunks, slices, words_per_slice, fixed_bits, shifts,
                           reinterpret_cast<unsigned long long*>(words));
    });
    BSI_LAUNCH_CHECK("shift_pack_kernel");
    return BSI_OK;
}

extern "C" int bsi_hip_pack_bits_batch(const int64_t* ints, int64_t Q, int64_t d, int slices, int words_per_slice,
                                       uint64_t* words, void* stream) {
    if (int rc = check_pack_args(Q, d, slices, words_per_slice)) return rc;
    if (Q == 0) return BSI_OK;
    BSI_REQUIRE(ints && words, "null pointer");
    const int groups = (words_per_slice + 3) / 4;
    RoundedFromInts src{reinterpret_cast<const long long*>(ints)};
    launch((shift_pack_kernel<RoundedFromInts, false>), dim3(grid_for(Q * groups)), dim3(kBlock), 0,
                       as_stream(stream), src, Q, d, 0, slices, words_per_slice, 0, nullptr,
                       reinterpret_cast<unsigned long long*>(words));
    BSI_LAUNCH_CHECK("shift_pack_kernel");
    return BSI_OK;
}

// ---- decimal mode (no fixed bits): the slice count follows the data ----

// One workgroup per row: largest |value| of the whole batch (atomic max into *max_abs, cleared by the
// launcher) and, per row, whether any value is negative.
__global__ __launch_bounds__(kBlock) void decimal_stats_kernel(const long long* __restrict__ ints, int64_t d,
                                                               unsigned long long* __restrict__ max_abs,
                                                               int* __restrict__ row_negative) {
    __shared__ unsigned long long smax[kBlock / BSI_WAVE];
    __shared__ int sneg[kBlock / BSI_WAVE];
    const int64_t q = blockIdx.x;
    const long long* row = ints + q * d;
    unsigned long long m = 0;
    int neg = 0;
    for (int64_t e = threadIdx.x; e < d; e += kBlock) {
        const long long v = row[e];
        const unsigned long long a = v < 0 ? 0ULL - static_cast<unsigned long long>(v) : static_cast<unsigned long long>(v);
        m = a > m ? a : m;
        neg |= v < 0;
    }
#pragma unroll
    for (int off = BSI_WAVE / 2; off > 0; off >>= 1) {
        const unsigned long long o = __shfl_xor(m, off, BSI_WAVE);
        m = o > m ? o : m;
        neg |= __shfl_xor(neg, off, BSI_WAVE);
    }
    const int wave = threadIdx.x / BSI_WAVE;
    if ((threadIdx.x & (BSI_WAVE - 1)) == 0) {
        smax[wave] = m;
        sneg[wave] = neg;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kBlock / BSI_WAVE; ++w) {
            m = smax[w] > m ? smax[w] : m;
            neg |= sneg[w];
        }
        row_negative[q] = neg;
        if (m != 0) atomicMax(max_abs, m);
    }
}

__global__ void clear_u64_kernel(unsigned long long* p) { *p = 0ULL; }

extern "C" int bsi_hip_decimal_stats(const int64_t* ints, int64_t Q, int64_t d, uint64_t* max_abs,
                                     int32_t* row_negative, void* stream) {
    BSI_REQUIRE(Q >= 0 && d >= 0, "negative size");
    BSI_REQUIRE(max_abs != nullptr, "null pointer");
    BSI_REQUIRE(Q <= 0x7fffffffLL, "too many rows for one launch");
    launch(clear_u64_kernel, dim3(1), dim3(1), 0, as_stream(stream),
                       reinterpret_cast<unsigned long long*>(max_abs));
    BSI_LAUNCH_CHECK("clear_u64_kernel");
    if (Q == 0) return BSI_OK;
    BSI_REQUIRE(row_negative != nullptr && (ints != nullptr || d == 0), "null pointer");
    launch(decimal_stats_kernel, dim3(static_cast<unsigned>(Q)), dim3(kBlock), 0, as_stream(stream),
                       reinterpret_cast<const long long*>(ints), d, reinterpret_cast<unsigned long long*>(max_abs),
                       row_negative);
    BSI_LAUNCH_CHECK("decimal_stats_kernel");
    return BSI_OK;
}

std::atomic<int> bsi::g_build_items{0};

// Whether rows of d elements at x can be loaded a quad at a time.
static bool quads_aligned(const void* x, int dtype, int64_t d) {
    return d % 4 == 0 && (reinterpret_cast<uintptr_t>(x) & (dtype == BSI_DTYPE_F32 ? 15 : 7)) == 0;
}
#define BSI_DISPATCH_BOOL(cond, name, ...)                        \
    if (cond) { constexpr bool name = true; __VA_ARGS__; }        \
    else { constexpr bool name = false; __VA_ARGS__; }

extern "C" int bsi_hip_build_fixed(const void* x, int dtype, int64_t Q, int64_t d, int decimal_places, int fixed_bits,
                                   int chunk_scale, float clip_k, uint64_t* words, int32_t* shifts, float* scales,
                                   int8_t* ints8, void* stream) {
    BSI_REQUIRE(Q >= 0 && d >= 0, "negative size");
    BSI_REQUIRE(fixed_bits >= 2 && fixed_bits <= 63, "fixed_bits must be in [2, 63]");
    BSI_REQUIRE(ints8 == nullptr || fixed_bits <= 8, "int8 output needs fixed_bits <= 8");
    if (Q == 0 || d == 0) return BSI_OK;
    const int W = static_cast<int>((d + 63) / 64);
    const int chunks = static_cast<int>((d + 255) / 256);
    const double dec_scale = pow(10.0, static_cast<double>(decimal_places));
    const unsigned scale_int = integer_decimal_scale(dec_scale);
    const int64_t items = Q * chunks;
    // The register-resident kernels quantise in float32: 10^dec an integer of at most 127 (0 to 2 decimal places), at most
    // 8 slices, no clipping; their item numbers are 32-bit.
    const bool fast = scale_int != 0 && fixed_bits <= 8 && !(clip_k > 0.0f) && items <= 0x7fffff00LL && Q <= 0x7fffffffLL;
    BSI_REQUIRE(x && scales && (shifts || fast) && (words || (fast && ints8)), "null pointer");
    const float scale = static_cast<float>(scale_int);
    unsigned long long* const words64 = reinterpret_cast<unsigned long long*>(words);
    hipStream_t st = as_stream(stream);
    if (fast && chunk_scale && W % 4 == 0) {
#define BSI_LAUNCH_FAST(N)                                                                                                 \
    BSI_DISPATCH_DTYPE(dtype, BSI_DISPATCH_BOOL(quads_aligned(x, dtype, d), kVec, BSI_DISPATCH_BOOL(words != nullptr, kPlanes, \
        launch((build_fixed_chunk_fast_kernel<T, N, kVec, kPlanes>), dim3(grid_for((items + (N) - 1) / (N))),  \
                           dim3(kBlock), 0, st, static_cast<const T*>(x), static_cast<unsigned>(items), d,                 \
                           static_cast<unsigned>(chunks), fixed_bits, W, dec_scale, scale, words64, shifts, scales, ints8))))
        // Several items a wave share its prologue and put their loads in flight together: worth it once every SIMD has its
        // eight waves without (16384 items: 6.5 us with one each, 6.0 with two, 6.3 with four; 65536: 18.1, 15.6, 15.4).
        int per_wave = g_build_items.load(std::memory_order_relaxed);
        if (per_wave == 0) per_wave = items >= 32768 ? 4 : (items >= 16384 ? 2 : 1);
        if (per_wave == 8) { BSI_LAUNCH_FAST(8); }
        else if (per_wave == 4) { BSI_LAUNCH_FAST(4); }
        else if (per_wave == 2) { BSI_LAUNCH_FAST(2); }
        else { BSI_LAUNCH_FAST(1); }
#undef BSI_LAUNCH_FAST
        BSI_LAUNCH_CHECK("build_fixed_chunk_fast_kernel");
    } else if (fast && !chunk_scale) {
        BSI_DISPATCH_DTYPE(dtype, BSI_DISPATCH_BOOL(quads_aligned(x, dtype, d), kVec, BSI_DISPATCH_BOOL(words != nullptr, kPlanes,
            launch((build_fixed_row_fast_kernel<T, kVec, kPlanes>), dim3(static_cast<unsigned>(Q)), dim3(kBlock), 0, st,
                               static_cast<const T*>(x), d, chunks, fixed_bits, W, dec_scale, scale, words64, shifts, scales,
                               ints8))))
        BSI_LAUNCH_CHECK("build_fixed_row_fast_kernel");
    } else if (chunk_scale) {
        BSI_REQUIRE(words != nullptr, "null pointer");
        BSI_DISPATCH_DTYPE(dtype, launch(build_fixed_chunk_kernel<T>, dim3(grid_for(items)), dim3(kBlock), 0, st,
                                                     static_cast<const T*>(x), Q, d, chunks, fixed_bits, W, dec_scale, clip_k,
                                                     words64, shifts, scales, ints8));
        BSI_LAUNCH_CHECK("build_fixed_chunk_kernel");
    } else {
        BSI_DISPATCH_DTYPE(dtype, launch(build_fixed_row_kernel<T>, dim3(static_cast<unsigned>(Q)), dim3(kBlock), 0,
                                                     st, static_cast<const T*>(x), Q, d, fixed_bits, W, dec_scale, clip_k,
                                                     words64, shifts, scales, ints8));
        BSI_LAUNCH_CHECK("build_fixed_row_kernel");
    }
    return BSI_OK;
}

extern "C" int bsi_hip_build_fixed_keys(const void* x, int dtype, int64_t R, int64_t d, int decimal_places, int fixed_bits,
                                        uint64_t* tiled, int8_t* image, int32_t* shifts, float* slice_weights, void* stream) {
    BSI_REQUIRE(R >= 0 && d >= 1, "bad shape");
    const unsigned scale_int = integer_decimal_scale(pow(10.0, static_cast<double>(decimal_places)));
    if (scale_int == 0 || fixed_bits < 2 || fixed_bits > 8)
        return fail(BSI_ERR_UNSUPPORTED, "the one-launch key build takes 2 to 8 bits and 0 to 2 decimal places (got %d and %d)",
                    fixed_bits, decimal_places);
    if (R == 0) return BSI_OK;
    BSI_REQUIRE(x && tiled && image && shifts && slice_weights, "null pointer");
    BSI_REQUIRE((R + kKeyRows - 1) / kKeyRows <= 0x7fffffffLL, "too many rows for one launch");
    const int chunks = static_cast<int>((d + 255) / 256);
    // Rows of up to 32 chunks stay in registers whole.  kHeld is the next of 8, 16 and 32, kLoads what the rest of the 64
    // registers takes in flight (32 chunks, 8192 x 5120 bfloat16 with plain stores: 2, 4, 8 loads 44, 31, 34 us).
    const int64_t tiles = (R + kKeyRows - 1) / kKeyRows;
#define BSI_KEYS(kHeld, kLoads, kOnce)                                                                                              \
    BSI_DISPATCH_DTYPE(dtype, BSI_DISPATCH_BOOL(quads_aligned(x, dtype, d), kVec,                                             \
        launch((build_keys_fast_kernel<T, kVec, kHeld, kLoads, kVec && kOnce>), dim3(static_cast<unsigned>(tiles)),                 \
               dim3(kKeyRows * BSI_WAVE), 0, as_stream(stream), static_cast<const T*>(x), R, d, chunks, fixed_bits,           \
               static_cast<double>(scale_int), static_cast<float>(scale_int),                                                \
               reinterpret_cast<unsigned long long*>(tiled), image, shifts, slice_weights)))
    const size_t row_bytes = static_cast<size_t>(d) * (dtype == BSI_DTYPE_F32 ? 4 : 2);
    const bool once = row_bytes % 128 == 0 && reinterpret_cast<uintptr_t>(x) % 128 == 0 &&
                      row_bytes * static_cast<size_t>(R) >= (chunks <= 16 ? kKeysOnceBytes : kKeysOnceLongBytes);
    if (chunks <= 8) { if (once) BSI_KEYS(8, 8, true) else BSI_KEYS(8, 8, false) }
    else if (chunks <= 16) { if (once) BSI_KEYS(16, 8, true) else BSI_KEYS(16, 8, false) }
    else { if (once) BSI_KEYS(32, 4, true) else BSI_KEYS(32, 4, false) }
#undef BSI_KEYS
    BSI_LAUNCH_CHECK("build_keys_fast_kernel");
    return BSI_OK;
}
