// The scalar entry points' one query against prebuilt decimal keys, in one launch: every workgroup builds the query for
// itself, in LDS.
#include "bsi_ewah_device.h"

#include <chrono>

namespace bsi {

constexpr int kScalarBlock = 512, kScalarWaves = kScalarBlock / BSI_WAVE;
constexpr int64_t kScalarMaxElems = 16384;  // 64 planes of it fill 128 KiB of LDS; a longer vector takes the batched builder
constexpr int kScalarMaxGroups = 512;       // two workgroups for each CU; more rows are looped over
constexpr unsigned long long kScalarPending = 0xFFF8DEADFFFFBEEFULL;  // a NaN no score has, and no count or clock value

__device__ __forceinline__ void store_host(unsigned long long* p, unsigned long long v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// out[r] = sum_{i,j,w} popcount(A[i, w] & B[r, j, w]) * Aw[i] * Bw[r, j], exact in float64 while below 2^53, where A are the
// planes of the decimal build of x (round half away from zero of x * 10^dec, the slice count from the largest magnitude).
// host: {slices, whether a value is negative, words of the stored form, run-length coded slices}, three clock values of
// every workgroup (begin, query built, end), then the R scores: pinned memory, each word stored once, so that the host sees
// from the words themselves that all have come and waits for no event.
// kLanes lanes share a key row, a word each.  A lane puts its popcounts together over the query's slices in integers (two
// v_bcnt and one shift a pair of slices), four key slices at a time, and multiplies by the key's weights once.  The last
// workgroup measures the stored form (density flag and EWAH length of every slice) instead of rows.
// Bound by latency: the first key words are requested before the query is built.  The build costs every workgroup 2 us and
// saves the launch of its own, with one busy CU, that it was before (9.0 + 6.8 us for 2048 elements against 1024 keys).
template <int kLanes>
__global__ __launch_bounds__(kScalarBlock) void scalar_query_dot_kernel(const float* __restrict__ x, int d, int W, double dec_scale,
                                                                        double threshold, const unsigned long long* __restrict__ B,
                                                                        const float* __restrict__ Bw, int Sb, int R,
                                                                        unsigned long long* __restrict__ host) {
    extern __shared__ unsigned long long As[];  // [slices][W]
    constexpr int kRows = kScalarBlock / kLanes;
    constexpr int kAhead = 8;                   // key slices requested up front
    constexpr int kHeld = 8;                    // words of the query a wave keeps in registers between its two passes
    __shared__ unsigned long long smax[kScalarWaves];
    __shared__ int sneg[kScalarWaves];
    __shared__ double scores[kRows];
    const unsigned long long began = wall_clock64();
    const int tid = threadIdx.x, lane = tid & (BSI_WAVE - 1), wave = tid >> 6;
    const bool measures = blockIdx.x == gridDim.x - 1;
    const int l = tid % kLanes, r0 = blockIdx.x * kRows + tid / kLanes;
    unsigned long long ahead[kAhead];
    {
        const int r = r0 < R ? r0 : R - 1, w = l < W ? l : W - 1;
#pragma unroll
        for (int j = 0; j < kAhead; ++j)
            ahead[j] = B[(static_cast<size_t>(r) * Sb + (j < Sb ? j : Sb - 1)) * W + w];
    }

    // the query: largest magnitude, then its planes
    auto value = [&](int w) {
        const int e = w * BSI_WAVE + lane;
        const float f = x[e < d ? e : d - 1];
        return e < d ? round_scaled(f, dec_scale) : 0LL;
    };
    long long held[kHeld];
    unsigned long long m = 0ULL;
    int neg = 0;
    auto look = [&](long long v) {
        const unsigned long long a = uabs_ll(v);
        m = a > m ? a : m;
        neg |= v < 0;
    };
#pragma unroll
    for (int k = 0; k < kHeld; ++k) held[k] = value(wave + k * kScalarWaves);  // past the vector: zeros
#pragma unroll
    for (int k = 0; k < kHeld; ++k) look(held[k]);
    for (int w = wave + kHeld * kScalarWaves; w < W; w += kScalarWaves) look(value(w));
    m = wave_max_u64(m);
    neg = __any(neg) ? 1 : 0;
    if (lane == 0) {
        smax[wave] = m;
        sneg[wave] = neg;
    }
    __syncthreads();
    m = 0ULL;
    neg = 0;
#pragma unroll
    for (int w = 0; w < kScalarWaves; ++w) {
        m = smax[w] > m ? smax[w] : m;
        neg |= sneg[w];
    }
    int S = m == 0ULL ? 2 : 64 - __clzll(static_cast<long long>(m)) + 2;  // the decimal builder's rule (bsi_vector_cuda.cpp:746-754)
    if (S > 64) S = 64;
    S = __builtin_amdgcn_readfirstlane(S);
    auto slice = [&](long long v, int w) {
        unsigned long long mine = 0ULL;
        for (int s = 0; s < S; ++s) {
            const unsigned long long word = __ballot((static_cast<unsigned long long>(v) >> s) & 1ULL);
            if (lane == s) mine = word;
        }
        if (lane < S) As[static_cast<size_t>(lane) * W + w] = mine;
    };
#pragma unroll
    for (int k = 0; k < kHeld; ++k)
        if (wave + k * kScalarWaves < W) slice(held[k], wave + k * kScalarWaves);
    for (int w = wave + kHeld * kScalarWaves; w < W; w += kScalarWaves) slice(value(w), w);
    __syncthreads();
    const unsigned long long built = wall_clock64();
    unsigned long long* const stamps = host + 4 + 3 * static_cast<size_t>(blockIdx.x);

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
            store_host(host + 1, static_cast<unsigned long long>(neg));
            store_host(host + 2, words);
            store_host(host + 3, static_cast<unsigned long long>(coded));
        }
    } else {
        unsigned long long* const out = host + 4 + 3 * static_cast<size_t>(gridDim.x);
        const int stride = (gridDim.x - 1) * kRows;
        for (int rb = blockIdx.x * kRows; rb < R; rb += stride) {
            const int r = rb + tid / kLanes;
            double acc = 0.0;
            auto four = [&](const unsigned long long (&b)[4], int w, int j0) {
                double part[4];
                auto combine = [&](auto zero) {
                    decltype(zero) t[4] = {zero, zero, zero, zero};
                    for (int i = S - 1; i >= 0; --i) {
                        const unsigned long long a = As[i * W + w];
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            const int c = __popcll(a & b[u]);
                            t[u] = t[u] * 2 + ((neg && i == S - 1) ? -c : c);
                        }
                    }
#pragma unroll
                    for (int u = 0; u < 4; ++u) part[u] = static_cast<double>(t[u]);
                };
                if (S <= 24) combine(0);              // 64 * 2^24 < 2^31
                else if (S <= 56) combine(0LL);       // 64 * 2^56 < 2^63
                else combine(0.0);
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (j0 + u < Sb) acc += part[u] * static_cast<double>(Bw[static_cast<size_t>(r) * Sb + j0 + u]);
            };
            if (r < R) {
                const unsigned long long* row = B + static_cast<size_t>(r) * Sb * W;
                for (int w = l; w < W; w += kLanes) {
                    const bool first = rb == static_cast<int>(blockIdx.x) * kRows && w == l;
                    for (int j0 = 0; j0 < Sb; j0 += 4) {
                        unsigned long long b[4];
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            if (first && j0 < kAhead) b[u] = j0 == 0 ? ahead[u] : ahead[4 + u];
                            else b[u] = row[static_cast<size_t>(j0 + u < Sb ? j0 + u : Sb - 1) * W + w];
                        }
                        four(b, w, j0);
                    }
                }
            }
#pragma unroll
            for (int off = kLanes / 2; off > 0; off >>= 1) acc += __shfl_xor(acc, off, BSI_WAVE);
            if (l == 0) scores[tid / kLanes] = acc;
            __syncthreads();
            if (tid < kRows && rb + tid < R) store_host(out + rb + tid, static_cast<unsigned long long>(__double_as_longlong(scores[tid])));
            __syncthreads();
        }
    }
    if (tid == 0) {
        store_host(stamps, began);
        store_host(stamps + 1, built);
        store_host(stamps + 2, wall_clock64());
    }
}

static int scalar_lanes(int64_t d) {  // the lanes of a row cover its words where they can
    const int64_t W = (d + 63) / 64;
    return W > 32 ? 64 : (W > 16 ? 32 : 16);
}
static int64_t scalar_groups(int64_t d, int64_t R) {
    const int rows = kScalarBlock / scalar_lanes(d);
    const int64_t groups = (R + rows - 1) / rows;
    return 1 + (groups < kScalarMaxGroups ? groups : kScalarMaxGroups);
}

}  // namespace bsi

using namespace bsi;

extern "C" int64_t bsi_hip_scalar_query_max_elems(void) { return kScalarMaxElems; }

extern "C" int64_t bsi_hip_scalar_query_host_words(int64_t d, int64_t R) { return 4 + 3 * scalar_groups(d, R) + R; }

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
    const int64_t groups = scalar_groups(d, R), words = bsi_hip_scalar_query_host_words(d, R);
    volatile unsigned long long* const host = reinterpret_cast<volatile unsigned long long*>(pinned);
    for (int64_t i = 0; i < words; ++i) host[i] = kScalarPending;
    std::atomic_thread_fence(std::memory_order_seq_cst);
#define BSI_SCALAR_DOT(L)                                                                                                  \
    {                                                                                                                      \
        static LdsOptIn once;                                                                                              \
        lds_opt_in(once, reinterpret_cast<const void*>(&scalar_query_dot_kernel<L>), 64 * 256 * 8);                        \
        launch(scalar_query_dot_kernel<L>, dim3(static_cast<unsigned>(groups)), dim3(kScalarBlock), static_cast<size_t>(64) * W * 8, \
               st, x, static_cast<int>(d), W, pow(10.0, static_cast<double>(decimal_places)), threshold,                   \
               reinterpret_cast<const unsigned long long*>(B), Bw, Sb, static_cast<int>(R),                                \
               reinterpret_cast<unsigned long long*>(pinned));                                                             \
    }
    const int lanes = scalar_lanes(d);
    if (lanes == 64) BSI_SCALAR_DOT(64)
    else if (lanes == 32) BSI_SCALAR_DOT(32)
    else BSI_SCALAR_DOT(16)
#undef BSI_SCALAR_DOT
    BSI_LAUNCH_CHECK("scalar_query_dot_kernel");
    // The words come while the kernel still runs; the stream is waited for only if they are long in coming.
    const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(500);
    bool waited = false;
    auto word = [&](int64_t i) {
        while (host[i] == kScalarPending && !waited) {
            if (std::chrono::steady_clock::now() > until) {
                waited = true;
                return hipStreamSynchronize(st);
            }
        }
        return hipSuccess;
    };
    for (int64_t i = 0; i < words; ++i) BSI_HIP_CHECK(word(i));
    const volatile unsigned long long* const stamps = host + 4;
    unsigned long long began = stamps[0], built = stamps[1], ended = stamps[2];
    for (int64_t g = 1; g < groups; ++g) {
        if (stamps[3 * g] < began) began = stamps[3 * g];
        if (stamps[3 * g + 1] > built) built = stamps[3 * g + 1];
        if (stamps[3 * g + 2] > ended) ended = stamps[3 * g + 2];
    }
    const double ns = 1.0e6 / static_cast<double>(clock_khz.load(std::memory_order_relaxed));
    *build_ns = static_cast<int64_t>(static_cast<double>(built - began) * ns);
    *dot_ns = static_cast<int64_t>(static_cast<double>(ended - built) * ns);
    for (int i = 0; i < 4; ++i) info[i] = static_cast<int64_t>(host[i]);
    const volatile double* const scores = reinterpret_cast<const volatile double*>(host + 4 + 3 * groups);
    for (int64_t r = 0; r < R; ++r) out[r] = scores[r] / divisor;
    return BSI_OK;
}
