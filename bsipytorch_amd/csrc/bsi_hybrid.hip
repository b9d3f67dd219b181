// Query batches kept as EWAH streams: the fixed-bit build with the measurement of every slice's stream in the same launch,
// and the emit pass that finds its own offsets.
#include "bsi_ewah_device.h"
#include "bsi_quant_device.h"

namespace bsi {

constexpr int kHybridBlock = 512, kHybridWaves = kHybridBlock / BSI_WAVE;
constexpr int kHybridMaxWords = 1024;    // a slice: eight of them fill 64 KiB of LDS
constexpr int kHybridMaxSlices = 8192;   // of the batch: what the emit pass sums up per workgroup

// One workgroup per row.  Its waves quantise a chunk each at a time (bsi_quant_device.h) and leave the planes in LDS; from
// there they go to memory in one contiguous run, and a wave for each slice counts and measures it: density flag and stream
// length.  The host (pinned memory, system scope) gets the length of every slice or, host_rows, of a whole row: it waits for
// the lengths and not for the kernel, and every word on the way is a write over the bus here and a cold line there.
// Bound by latency (load, two barriers, the codec's ballots).  64 rows of 2048: 4.8 us, against 2.9 for the build, 4.0 for
// the measurement and 2.6 for the offsets in launches of their own.  Seven lengths a row and one: 512 x 2048 12.2 us and 6; a
// batch with its dot against 2048 keys 61 us and 38, 64 x 2048 38 and 31 (with the codec's loads beside each other).
template <typename T, bool kVec>
__global__ __launch_bounds__(kHybridBlock) void build_measure_kernel(const T* __restrict__ x, int64_t d, int chunks, int slices, int W,
                                                                     int row_scale, double dec_scale, float scale, double threshold,
                                                                     unsigned long long* __restrict__ words, float* __restrict__ scales,
                                                                     float* __restrict__ weights, int* __restrict__ flags,
                                                                     int* __restrict__ lens, int* __restrict__ lens_host, int host_rows) {
    extern __shared__ __attribute__((aligned(16))) uint32_t planes[];  // [slices][2 W]
    constexpr int kHeld = 4;
    __shared__ unsigned smax[kHybridWaves];
    __shared__ unsigned long long smax64[kHybridWaves];
    __shared__ unsigned row_sum;  // slices measured << 24 | their lengths (at most 8 x 1025 words)
    const int lane = threadIdx.x & (BSI_WAVE - 1);
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t row = blockIdx.x;
    const T* xrow = x + row * d;
    const ChunkLane cl = chunk_lane(lane);
    const QuantRange range = quant_range(slices);
    if (threadIdx.x == 0) row_sum = 0u;  // ahead of the barrier behind the planes
    float v[kHeld][4];
#pragma unroll
    for (int j = 0; j < kHeld; ++j) load_chunk_quad<T, kVec>(xrow, d, wid + j * kHybridWaves, cl, v[j]);  // past the row: zeros

    int row_shift = 0;
    bool row_wide = false;
    if (row_scale) {
        unsigned mx = 0u;
#pragma unroll
        for (int j = 0; j < kHeld; ++j) {
            const unsigned m = quad_max_bits(v[j]);
            mx = m > mx ? m : mx;
        }
        for (int c = wid + kHeld * kHybridWaves; c < chunks; c += kHybridWaves) {
            float t[4];
            load_chunk_quad<T, kVec>(xrow, d, c, cl, t);
            const unsigned m = quad_max_bits(t);
            mx = m > mx ? m : mx;
        }
        mx = wave_max_u32(mx);
        if (lane == 0) smax[wid] = mx;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < kHybridWaves; ++w) mx = smax[w] > mx ? smax[w] : mx;
        row_wide = mx >= kQuantWideBits;
        row_shift = quant_shift(mx, scale, slices);
        if (row_wide) {
            unsigned long long m64 = 0ULL;
            for (int c = wid; c < chunks; c += kHybridWaves) {
                float t[4];
                load_chunk_quad<T, kVec>(xrow, d, c, cl, t);
                const unsigned long long m = quad_max_wide(t, dec_scale);
                m64 = m > m64 ? m : m64;
            }
            m64 = wave_max_u64(m64);
            if (lane == 0) smax64[wid] = m64;
            __syncthreads();
            for (int w = 0; w < kHybridWaves; ++w) m64 = smax64[w] > m64 ? smax64[w] : m64;
            row_shift = compute_shift(m64, 0.0, 1, slices, 0.0f);
        }
        if (static_cast<int>(threadIdx.x) < slices) {
            const float w = static_cast<float>(1ULL << row_shift) * static_cast<float>(1 << threadIdx.x);
            weights[row * slices + threadIdx.x] = static_cast<int>(threadIdx.x) == slices - 1 ? -w : w;
        }
        if (threadIdx.x == 0) scales[row] = static_cast<float>(1ULL << row_shift);
    }
    auto emit = [&](int c, const float (&t)[4]) {
        int shift = row_shift;
        bool wide = row_wide;
        if (!row_scale) {
            const unsigned mx = wave_max_u32(quad_max_bits(t));
            wide = mx >= kQuantWideBits;
            shift = wide ? compute_shift(wave_max_u64(quad_max_wide(t, dec_scale)), 0.0, 1, slices, 0.0f) : quant_shift(mx, scale, slices);
            if (lane == 0) scales[row * chunks + c] = static_cast<float>(1ULL << shift);
        }
        const uint32_t image = chunk_image_dword(wide ? quantise_quad_wide(t, dec_scale, shift, slices)
                                                      : quantise_quad<T>(t, scale, shift, range), cl);
        const uint32_t plane = chunk_plane_dword(image, cl);
        const int sl = (lane & 7) - (8 - slices), unit = c * 8 + (lane >> 3);
        if (sl >= 0 && unit < 2 * W) planes[sl * 2 * W + unit] = plane;
    };
#pragma unroll
    for (int j = 0; j < kHeld; ++j)
        if (wid + j * kHybridWaves < chunks) emit(wid + j * kHybridWaves, v[j]);
    for (int c = wid + kHeld * kHybridWaves; c < chunks; c += kHybridWaves) {
        float t[4];
        load_chunk_quad<T, kVec>(xrow, d, c, cl, t);
        emit(c, t);
    }
    __syncthreads();

    const unsigned long long* const staged = reinterpret_cast<const unsigned long long*>(planes);
    for (int s = wid; s < slices; s += kHybridWaves) {
        const unsigned long long* base = staged + static_cast<size_t>(s) * W;
        unsigned long long count = 0ULL;
        for (int w = lane; w < W; w += BSI_WAVE) count += static_cast<unsigned long long>(__popcll(base[w]));
        const int flag = compress_flag(wave_sum_u64(count), W, threshold);
        const int n = flag ? static_cast<int>(ewah_encode_wave(base, W, 1, nullptr, lane)) : W + 1;
        if (lane == 0) {
            if (host_rows) {
                const unsigned before = atomicAdd(&row_sum, 1u << 24 | static_cast<unsigned>(n));
                if (before >> 24 == static_cast<unsigned>(slices) - 1)
                    __hip_atomic_store(lens_host + row, static_cast<int>(before & 0xffffffu) + n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            } else {
                __hip_atomic_store(lens_host + row * slices + s, n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            }
            flags[row * slices + s] = flag;
            lens[row * slices + s] = n;
        }
    }
    for (int i = threadIdx.x; i < slices * W; i += kHybridBlock) words[row * slices * W + i] = staged[i];
}

// Four slices a workgroup, a wave each.  A workgroup sums the lengths of all slices before its own (32 KiB at most, from the
// L2): cheaper than a launch for the offsets.  The slice's first 64 words and its flag are asked for ahead of the sum.
constexpr int kEmitBlock = 256, kEmitWaves = kEmitBlock / BSI_WAVE;
__global__ __launch_bounds__(kEmitBlock) void ewah_emit_at_kernel(const unsigned long long* __restrict__ words, int S, int W,
                                                                  const int* __restrict__ flags, const int* __restrict__ lens,
                                                                  long long* __restrict__ off, unsigned long long* __restrict__ out) {
    __shared__ int sums[kEmitWaves];
    const int lane = threadIdx.x & (BSI_WAVE - 1);
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int first = blockIdx.x * kEmitWaves;  // a multiple of 4, as the lengths are read
    const int s = first + wid;
    const unsigned long long* const base = words + static_cast<size_t>(s) * W;
    const unsigned long long head = s < S && lane < W ? base[lane] : 0ULL;  // beside the lengths, not behind them
    const int flag = s < S ? flags[s] : 0;
    const int4* const quads = reinterpret_cast<const int4*>(lens);
    int sum = 0;
    for (int i = threadIdx.x; i < first / 4; i += kEmitBlock) {
        const int4 q = quads[i];
        sum += q.x + q.y + q.z + q.w;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, BSI_WAVE);
    if (lane == 0) sums[wid] = sum;
    __syncthreads();
    if (s >= S) return;
    long long at = 0;
    for (int w = 0; w < kEmitWaves; ++w) at += sums[w];
    for (int w = 0; w < wid; ++w) at += lens[first + w];
    if (lane == 0) off[s] = at;
    ewah_encode_wave(base, W, flag, out + at, lane, head);
}

}  // namespace bsi

using namespace bsi;

static int build_measure(const void* x, int dtype, int64_t Q, int64_t d, int decimal_places, int fixed_bits, int chunk_scale,
                         double threshold, uint64_t* words, float* scales, float* weights, int32_t* flags, int32_t* lens,
                         int32_t* lens_host, int host_rows, void* stream) {
    const double dec_scale = pow(10.0, static_cast<double>(decimal_places));
    const unsigned scale_int = integer_decimal_scale(dec_scale);
    BSI_REQUIRE(Q >= 1 && d >= 1 && fixed_bits >= 2 && fixed_bits <= 8, "bad shape");
    const int64_t W = (d + 63) / 64;
    if (scale_int == 0 || W > kHybridMaxWords || Q * fixed_bits > kHybridMaxSlices)
        return fail(BSI_ERR_UNSUPPORTED, "the build with measurement takes 0 to 2 decimal places, %d words a slice and %d slices",
                    kHybridMaxWords, kHybridMaxSlices);
    BSI_REQUIRE(x && words && scales && flags && lens && lens_host && (chunk_scale || weights), "null pointer");
    BSI_REQUIRE(!chunk_scale || W % 4 == 0, "chunk scales need a multiple of 4 words per slice");
    const size_t esize = dtype == BSI_DTYPE_F32 ? 4 : 2;
    const bool vec = d % 4 == 0 && reinterpret_cast<uintptr_t>(x) % (4 * esize) == 0;
#define BSI_GO(T, V)                                                                                                        \
    launch((build_measure_kernel<T, V>), dim3(static_cast<unsigned>(Q)), dim3(kHybridBlock), static_cast<size_t>(fixed_bits * W * 8), \
           as_stream(stream), static_cast<const T*>(x), d, static_cast<int>((d + 255) / 256), fixed_bits, static_cast<int>(W), \
           chunk_scale ? 0 : 1, dec_scale, static_cast<float>(scale_int), threshold, reinterpret_cast<unsigned long long*>(words), scales, \
           weights, flags, lens, lens_host, host_rows)
    switch (dtype) {
        case BSI_DTYPE_F32: if (vec) BSI_GO(float, true); else BSI_GO(float, false); break;
        case BSI_DTYPE_F16: if (vec) BSI_GO(__half, true); else BSI_GO(__half, false); break;
        case BSI_DTYPE_BF16: if (vec) BSI_GO(__hip_bfloat16, true); else BSI_GO(__hip_bfloat16, false); break;
        default: return fail(BSI_ERR_INVALID, "unknown dtype code %d", dtype);
    }
#undef BSI_GO
    BSI_LAUNCH_CHECK("build_measure_kernel");
    return BSI_OK;
}

extern "C" int bsi_hip_build_measure(const void* x, int dtype, int64_t Q, int64_t d, int decimal_places, int fixed_bits, int chunk_scale,
                                     double threshold, uint64_t* words, float* scales, float* weights, int32_t* flags, int32_t* lens,
                                     int32_t* lens_host, void* stream) {
    return build_measure(x, dtype, Q, d, decimal_places, fixed_bits, chunk_scale, threshold, words, scales, weights, flags, lens, lens_host, 0, stream);
}

extern "C" int bsi_hip_build_measure_rows(const void* x, int dtype, int64_t Q, int64_t d, int decimal_places, int fixed_bits, int chunk_scale,
                                          double threshold, uint64_t* words, float* scales, float* weights, int32_t* flags, int32_t* lens,
                                          int32_t* row_lens_host, void* stream) {
    return build_measure(x, dtype, Q, d, decimal_places, fixed_bits, chunk_scale, threshold, words, scales, weights, flags, lens, row_lens_host, 1, stream);
}

extern "C" int bsi_hip_ewah_emit_at(const uint64_t* words, int S, int W, const int32_t* flags, const int32_t* lens, int64_t* off,
                                    uint64_t* out, void* stream) {
    BSI_REQUIRE(S >= 1 && S <= kHybridMaxSlices && W >= 1, "bad shape");
    BSI_REQUIRE(words && flags && lens && off && out && (reinterpret_cast<uintptr_t>(lens) & 15) == 0, "null or unaligned pointer");
    launch(ewah_emit_at_kernel, dim3(static_cast<unsigned>((S + kEmitWaves - 1) / kEmitWaves)), dim3(kEmitBlock), 0, as_stream(stream),
           reinterpret_cast<const unsigned long long*>(words), S, W, flags, lens, reinterpret_cast<long long*>(off),
           reinterpret_cast<unsigned long long*>(out));
    BSI_LAUNCH_CHECK("ewah_emit_at_kernel");
    return BSI_OK;
}
