// The scalar entry points' one query against prebuilt decimal keys, in one launch: every workgroup builds the query for
// itself, in LDS.
#include "bsi_ewah_device.h"
#include "bsi_quant_device.h"

#include <chrono>
#include <cstring>

namespace bsi {

constexpr int kScalarBlock = 512, kScalarWaves = kScalarBlock / BSI_WAVE;
constexpr int64_t kScalarMaxElems = 12288;  // 64 planes of it and the vector take 144 KiB of LDS; a longer one the batched builder
constexpr int kScalarMaxGroups = 512;       // two workgroups for each CU; more rows are looped over
constexpr int kScalarStamps = 16;           // workgroups that report their clock
constexpr unsigned long long kScalarPending = 0xFFF8DEADFFFFBEEFULL;  // a NaN no score has, and no count or clock value

__device__ __forceinline__ void store_host(unsigned long long* p, unsigned long long v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// out[r] = sum_{i,j,w} popcount(A[i, w] & B[r, j, w]) * Aw[i] * Bw[r, j] / divisor, the sum exact in float64 while below 2^53, where A are the
// planes of the decimal build of x (round half away from zero of x * 10^dec, the slice count from the largest magnitude).
// host: {slices, whether a value is negative, words of the stored form, run-length coded slices}, three clock values of
// kScalarStamps workgroups (begin, query built, end), then the R scores: pinned memory, each word stored once, so that the
// host sees from the words themselves that all have come and waits for no event.
// A wave takes a key row: kWords words by 64 / kWords parts of its slices.  A lane puts its popcounts together over the
// query's slices in integers (two v_and, two v_bcnt and a shift a pair of slices), three key slices at a time, and
// multiplies by the key's weights once.  The last workgroup measures the stored form (density flag and EWAH length of every
// slice) instead of rows.
// Bound by latency and by VALU issue in the slicing and the popcounts; the first key words are requested before the query is
// built.  Every workgroup building it costs less than the launch of its own, with one busy CU, that the build was before.
// 2048 elements against 1024 keys, by a kernel trace: 9.0 + 6.8 us in two launches, 6.6 us in this one (5.3 from the first
// workgroup's clock to the last's, 3.1 of them until the query is built).
template <int kWords>
__global__ __launch_bounds__(kScalarBlock) void scalar_query_dot_kernel(const float* __restrict__ x, int d, int W, double dec_scale,
                                                                        int narrow, double threshold, const unsigned long long* __restrict__ B,
                                                                        const float* __restrict__ Bw, int Sb, int R, double divisor,
                                                                        unsigned long long* __restrict__ host) {
    extern __shared__ __attribute__((aligned(16))) unsigned long long As[];  // [64 slices][W], then x in whole chunks
    constexpr int kRows = kScalarWaves, kParts = BSI_WAVE / kWords;
    constexpr int kTogether = 3, kAhead = 2 * kTogether;  // key slices of a lane taken together, requested up front
    float* const xs = reinterpret_cast<float*>(As + static_cast<size_t>(64) * W);
    __shared__ uint2 smax[kScalarWaves];
    __shared__ double scores[kRows];
    const unsigned long long began = wall_clock64();
    const int tid = threadIdx.x, lane = tid & (BSI_WAVE - 1), wave = tid >> 6;
    const bool measures = blockIdx.x == gridDim.x - 1;
    const int l = lane % kWords, part = lane / kWords, r0 = blockIdx.x * kRows + wave;
    // the vector into LDS, and its largest magnitude as float bits (the rounded magnitudes are in the same order; a NaN is
    // rounded to the largest one, and to a negative value); the loads of a CU return in order: these before the keys'
    unsigned m = 0u, mneg = 0u;
    const int chunks = (d + BSI_CHUNK_ELEMS - 1) / BSI_CHUNK_ELEMS;
    for (int e = tid; e < chunks * BSI_CHUNK_ELEMS; e += kScalarBlock) {
        const float f = e < d ? x[e] : 0.0f;
        xs[e] = f;
        const unsigned bits = __float_as_uint(f) & 0x7fffffffu;
        const unsigned nbits = f >= 0.0f ? 0u : bits;
        m = bits > m ? bits : m;
        mneg = nbits > mneg ? nbits : mneg;
    }
    unsigned long long ahead[kAhead];
    {
        const int r = r0 < R ? r0 : R - 1, w = l < W ? l : W - 1;
#pragma unroll
        for (int j = 0; j < kAhead; ++j)
            ahead[j] = B[(static_cast<size_t>(r) * Sb + (part + kParts * j < Sb ? part + kParts * j : Sb - 1)) * W + w];
    }
    m = wave_max_u32(m);
    mneg = wave_max_u32(mneg);
    if (lane == 0) smax[wave] = make_uint2(m, mneg);
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kScalarWaves; ++w) {
        m = smax[w].x > m ? smax[w].x : m;
        mneg = smax[w].y > mneg ? smax[w].y : mneg;
    }
    const unsigned long long largest = uabs_ll(round_scaled(__uint_as_float(m), dec_scale));
    const bool neg = uabs_ll(round_scaled(__uint_as_float(mneg), dec_scale)) != 0ULL;
    int S = largest == 0ULL ? 2 : 64 - __clzll(static_cast<long long>(largest)) + 2;  // the decimal builder's rule (bsi_vector_cuda.cpp:746-754)
    if (S > 64) S = 64;
    S = __builtin_amdgcn_readfirstlane(S);

    // its planes.  Where every |x| (and 10^dec: narrow) is in the float32 quantiser's range the magnitudes are 32-bit integers:
    // a wave takes a chunk of 256, and every byte of the integers goes through the builders' transposes (bsi_quant_device.h).
    if (narrow && m < kQuantWideBits) {
        const float scale = static_cast<float>(dec_scale);
        const ChunkLane cl = chunk_lane(lane);
        uint32_t* const As32 = reinterpret_cast<uint32_t*>(As);
        for (int c = wave; c < chunks; c += kScalarWaves) {
            const float4 f = *reinterpret_cast<const float4*>(xs + c * BSI_CHUNK_ELEMS + cl.quad);
            const float fs[4] = {f.x, f.y, f.z, f.w};
            uint32_t v[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int a = static_cast<int>(scaled_magnitude_f32<float>(fabsf(fs[k]), scale));
                v[k] = static_cast<uint32_t>(fs[k] < 0.0f ? -a : a);
            }
            const int unit = c * 8 + (lane >> 3);
            for (int s0 = 0; s0 < S; s0 += 8) {
                const uint32_t plane = chunk_plane_dword(chunk_image_dword(pack_low_bytes(v[0], v[1], v[2], v[3]), cl), cl);
                const int s = s0 + (lane & 7);
                if (s < S && unit < 2 * W) As32[s * 2 * W + unit] = plane;
#pragma unroll
                for (int k = 0; k < 4; ++k) v[k] >>= 8;
            }
        }
    } else {
        for (int w = wave; w < W; w += kScalarWaves) {
            const unsigned long long v = static_cast<unsigned long long>(round_scaled(xs[w * BSI_WAVE + lane], dec_scale));
            unsigned long long mine = 0ULL;
            for (int s = 0; s < S; ++s) {
                const unsigned long long word = __ballot((v >> s) & 1ULL);
                if (lane == s) mine = word;
            }
            if (lane < S) As[static_cast<size_t>(lane) * W + w] = mine;
        }
    }
    __syncthreads();
    const unsigned long long built = wall_clock64();
    const unsigned stamp = measures ? (gridDim.x < kScalarStamps ? gridDim.x : kScalarStamps) - 1 : blockIdx.x;
    unsigned long long* const stamps = host + 4 + 3 * stamp;

    if (measures) {
        __shared__ unsigned long long swords[kScalarWaves];
        __shared__ int scoded[kScalarWaves];
        unsigned long long words = 0ULL;
        int coded = 0;
        for (int s = wave; s < S; s += kScalarWaves) {
            const unsigned long long* base = As + static_cast<size_t>(s) * W;
            unsigned long long count = 0ULL;
            for (int w = lane; w < W; w += BSI_WAVE) count += static_cast<unsigned long long>(__popcll(base[w]));
            const int flag = compress_flag(wave_sum_u64(count), W, threshold);
            words += flag ? ewah_encode_wave(base, W, 1, nullptr, lane) : static_cast<unsigned long long>(W) + 1ULL;
            coded += flag;
        }
        if (lane == 0) {
            swords[wave] = words;
            scoded[wave] = coded;
        }
        __syncthreads();
        if (tid == 0) {
            words = 0ULL;
            coded = 0;
            for (int w = 0; w < kScalarWaves; ++w) {
                words += swords[w];
                coded += scoded[w];
            }
            store_host(host, static_cast<unsigned long long>(S));
            store_host(host + 1, neg ? 1ULL : 0ULL);
            store_host(host + 2, words);
            store_host(host + 3, static_cast<unsigned long long>(coded));
        }
    } else {
        unsigned long long* const out = host + 4 + 3 * (gridDim.x < kScalarStamps ? gridDim.x : kScalarStamps);
        const int stride = (gridDim.x - 1) * kRows;
        for (int rb = blockIdx.x * kRows; rb < R; rb += stride) {
            const int r = rb + wave;
            double acc = 0.0;
            if (r < R) {
                const unsigned long long* row = B + static_cast<size_t>(r) * Sb * W;
#pragma unroll 1
                for (int w = l; w < W; w += kWords) {
                    const bool first = rb == static_cast<int>(blockIdx.x) * kRows && w == l;
#pragma unroll 1
                    for (int i0 = 0; i0 * kParts < Sb; i0 += kTogether) {
                        unsigned long long b[kTogether];
#pragma unroll
                        for (int u = 0; u < kTogether; ++u) {
                            const int j = part + kParts * (i0 + u);
                            if (first && i0 < kAhead) b[u] = i0 == 0 ? ahead[u] : ahead[kTogether + u];
                            else b[u] = row[static_cast<size_t>(j < Sb ? j : Sb - 1) * W + w];
                        }
                        double part_sum[kTogether];
                        auto combine = [&](auto zero) {
                            decltype(zero) t[kTogether];
                            const unsigned long long top = As[(S - 1) * W + w];
#pragma unroll
                            for (int u = 0; u < kTogether; ++u) {
                                const int c = __popcll(top & b[u]);
                                t[u] = neg ? -c : c;
                            }
#pragma unroll 4
                            for (int i = S - 2; i >= 0; --i) {
                                const unsigned long long a = As[i * W + w];
#pragma unroll
                                for (int u = 0; u < kTogether; ++u) t[u] = t[u] * 2 + __popcll(a & b[u]);
                            }
#pragma unroll
                            for (int u = 0; u < kTogether; ++u) part_sum[u] = static_cast<double>(t[u]);
                        };
                        if (S <= 24) combine(0);              // 64 * 2^24 < 2^31
                        else if (S <= 56) combine(0LL);       // 64 * 2^56 < 2^63
                        else combine(0.0);
#pragma unroll
                        for (int u = 0; u < kTogether; ++u) {
                            const int j = part + kParts * (i0 + u);
                            if (j < Sb) acc += part_sum[u] * static_cast<double>(Bw[static_cast<size_t>(r) * Sb + j]);
                        }
                    }
                }
            }
#pragma unroll
            for (int off = BSI_WAVE / 2; off > 0; off >>= 1) acc += __shfl_xor(acc, off, BSI_WAVE);
            if (lane == 0) scores[wave] = acc;
            __syncthreads();
            if (tid < kRows && rb + tid < R) store_host(out + rb + tid, static_cast<unsigned long long>(__double_as_longlong(scores[tid] / divisor)));
            __syncthreads();
        }
    }
    if (tid == 0 && (measures || stamp < kScalarStamps - 1)) {
        store_host(stamps, began);
        store_host(stamps + 1, built);
        store_host(stamps + 2, wall_clock64());
    }
}

static int64_t scalar_groups(int64_t R) {
    const int64_t groups = (R + kScalarWaves - 1) / kScalarWaves;
    return 1 + (groups < kScalarMaxGroups ? groups : kScalarMaxGroups);
}

}  // namespace bsi

using namespace bsi;

extern "C" int64_t bsi_hip_scalar_query_max_elems(void) { return kScalarMaxElems; }

extern "C" int64_t bsi_hip_scalar_query_host_words(int64_t R) {
    const int64_t groups = scalar_groups(R);
    return 4 + 3 * (groups < kScalarStamps ? groups : kScalarStamps) + R;
}

extern "C" int bsi_hip_scalar_query_dot(const float* x, int64_t d, int decimal_places, double threshold, const uint64_t* B,
                                        const float* Bw, int Sb, int64_t R, double divisor, uint64_t* pinned, double* out,
                                        int64_t* info, int64_t* build_ns, int64_t* dot_ns, void* stream) {
    BSI_REQUIRE(d >= 1 && d <= kScalarMaxElems, "d must be in [1, %lld] (got %lld)", static_cast<long long>(kScalarMaxElems),
                static_cast<long long>(d));
    BSI_REQUIRE(R >= 1 && R <= (1 << 24) && Sb >= 1 && Sb <= 64, "bad shape");
    BSI_REQUIRE(x && B && Bw && pinned && out && info && build_ns && dot_ns, "null pointer");
    hipStream_t st = as_stream(stream);
    static std::atomic<int> clock_khz{0};  // the same for every GPU of this architecture
    if (clock_khz.load(std::memory_order_relaxed) == 0) {
        int dev = 0, khz = 0;
        BSI_HIP_CHECK(hipGetDevice(&dev));
        BSI_HIP_CHECK(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev));
        clock_khz.store(khz > 0 ? khz : 100000, std::memory_order_relaxed);
    }
    const int W = static_cast<int>((d + 63) / 64);
    const int64_t groups = scalar_groups(R), words = bsi_hip_scalar_query_host_words(R), stamped = (words - R - 4) / 3;
    volatile unsigned long long* const host = reinterpret_cast<volatile unsigned long long*>(pinned);
    for (int64_t i = 0; i < words; ++i) host[i] = kScalarPending;
    std::atomic_thread_fence(std::memory_order_seq_cst);
    const double dec_scale = pow(10.0, static_cast<double>(decimal_places));
    const int narrow = integer_decimal_scale(dec_scale) != 0 ? 1 : 0;
#define BSI_SCALAR_DOT(L)                                                                                                  \
    {                                                                                                                      \
        static LdsOptIn once;                                                                                              \
        lds_opt_in(once, reinterpret_cast<const void*>(&scalar_query_dot_kernel<L>), kScalarMaxElems * 12);                       \
        launch(scalar_query_dot_kernel<L>, dim3(static_cast<unsigned>(groups)), dim3(kScalarBlock), static_cast<size_t>(W) * 512 + static_cast<size_t>((W + 3) / 4) * 1024, \
               st, x, static_cast<int>(d), W, dec_scale, narrow, threshold,                   \
               reinterpret_cast<const unsigned long long*>(B), Bw, Sb, static_cast<int>(R), divisor,                       \
               reinterpret_cast<unsigned long long*>(pinned));                                                             \
    }
    if (W > 32) BSI_SCALAR_DOT(64)
    else if (W > 16) BSI_SCALAR_DOT(32)
    else BSI_SCALAR_DOT(16)
#undef BSI_SCALAR_DOT
    BSI_LAUNCH_CHECK("scalar_query_dot_kernel");
    // The words come while the kernel still runs; the stream is waited for only if they are long in coming.
    const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(500);
    bool waited = false;
    auto word = [&](int64_t i, unsigned long long& v) {
        while ((v = host[i]) == kScalarPending && !waited) {
            if (std::chrono::steady_clock::now() > until) {
                waited = true;
                const hipError_t status = hipStreamSynchronize(st);
                v = host[i];
                return status;
            }
        }
        return hipSuccess;
    };
    // The scores go to the caller as they come, divided on the GPU: a pass of divisions behind the last of them, over lines that have been
    // read before, was 1.5 us of a call of 1024 scores of 2048 elements (19.8, 18.3) and 4 of one of 4096 x 4096 (27.3, 23.1).
    unsigned long long v = 0ULL;
    for (int64_t r = 0; r < R; ++r) {
        BSI_HIP_CHECK(word(4 + 3 * stamped + r, v));
        std::memcpy(out + r, &v, sizeof v);
    }
    for (int64_t i = 0; i < 4 + 3 * stamped; ++i) BSI_HIP_CHECK(word(i, v));  // the clocks at the end come behind the scores
    const volatile unsigned long long* const stamps = host + 4;
    unsigned long long began = stamps[0], built = stamps[1], ended = stamps[2];
    for (int64_t g = 1; g < stamped; ++g) {
        if (stamps[3 * g] < began) began = stamps[3 * g];
        if (stamps[3 * g + 1] > built) built = stamps[3 * g + 1];
        if (stamps[3 * g + 2] > ended) ended = stamps[3 * g + 2];
    }
    const double ns = 1.0e6 / static_cast<double>(clock_khz.load(std::memory_order_relaxed));
    *build_ns = static_cast<int64_t>(static_cast<double>(built - began) * ns);
    *dot_ns = static_cast<int64_t>(static_cast<double>(ended - built) * ns);
    for (int i = 0; i < 4; ++i) info[i] = static_cast<int64_t>(host[i]);
    return BSI_OK;
}
