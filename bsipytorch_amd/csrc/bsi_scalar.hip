// The scalar entry points' one query against prebuilt decimal keys, in two launches and one wait: the query's slice count
// stays on the device between them.
#include "bsi_ewah_device.h"

namespace bsi {

constexpr int kScalarBlock = 1024, kScalarWaves = kScalarBlock / BSI_WAVE;
constexpr int64_t kScalarMaxElems = 16384;  // one workgroup quantises the vector; a longer one takes the batched builder

// Decimal build of one vector by one workgroup: round half away from zero of x * 10^dec, the slice count from the largest
// magnitude, the planes [S, W], and what the stored form of the slices takes (density flag, EWAH length).
// info: {slices, whether a value is negative, words of the stored form, run-length coded slices}.
// Bound by its serial phases (three barriers, a few dependent loads): 2048 elements take about 8 us, against nine
// launches and five waits of the batched builder and codec.
__global__ __launch_bounds__(kScalarBlock) void scalar_query_kernel(const float* __restrict__ x, int d, int W, double dec_scale,
                                                                    double threshold, unsigned long long* __restrict__ planes,
                                                                    long long* __restrict__ info, long long* __restrict__ info_host) {
    __shared__ unsigned long long smax[kScalarWaves];
    __shared__ int sneg[kScalarWaves];
    __shared__ unsigned long long swords[kScalarWaves];
    __shared__ int scoded[kScalarWaves];
    const int tid = threadIdx.x, lane = tid & (BSI_WAVE - 1), wave = tid >> 6;
    unsigned long long m = 0ULL;
    int neg = 0;
    for (int e = tid; e < d; e += kScalarBlock) {
        const long long v = round_scaled(x[e], dec_scale);
        const unsigned long long a = uabs_ll(v);
        m = a > m ? a : m;
        neg |= v < 0;
    }
    m = wave_max_u64(m);
    neg = __any(neg) ? 1 : 0;
    if (lane == 0) {
        smax[wave] = m;
        sneg[wave] = neg;
    }
    __syncthreads();
    m = 0ULL;
    neg = 0;
    for (int w = 0; w < kScalarWaves; ++w) {
        m = smax[w] > m ? smax[w] : m;
        neg |= sneg[w];
    }
    int S = m == 0ULL ? 2 : 64 - __clzll(static_cast<long long>(m)) + 2;  // the decimal builder's rule (bsi_vector_cuda.cpp:746-754)
    if (S > 64) S = 64;
    for (int w = wave; w < W; w += kScalarWaves) {
        const int e = w * BSI_WAVE + lane;
        const unsigned long long v = e < d ? static_cast<unsigned long long>(round_scaled(x[e], dec_scale)) : 0ULL;
        unsigned long long mine = 0ULL;
        for (int s = 0; s < S; ++s) {
            const unsigned long long word = __ballot((v >> s) & 1ULL);
            if (lane == s) mine = word;
        }
        if (lane < S) planes[static_cast<size_t>(lane) * W + w] = mine;
    }
    __syncthreads();  // the planes of the other waves are read below
    unsigned long long words = 0ULL;
    int coded = 0;
    for (int s = wave; s < S; s += kScalarWaves) {
        const unsigned long long* base = planes + static_cast<size_t>(s) * W;
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
        const long long v[4] = {S, neg, static_cast<long long>(words), coded};
        for (int i = 0; i < 4; ++i) info[i] = info_host[i] = v[i];
    }
}

// out[r] = sum_{i,j,w} popcount(A[i, w] & B[r, j, w]) * Aw[i] * Bw[r, j], exact in float64 while below 2^53, for one query
// whose slice count and signedness are in `info`.  kLanes lanes share a key row, a word each; the query's planes sit in
// LDS.  A lane puts its popcounts together over the query's slices in integers (two v_bcnt and one shift a pair of
// slices), four key slices at a time, and multiplies by the key's weights once.
template <int kLanes>
__global__ __launch_bounds__(256) void scalar_dot_kernel(const unsigned long long* __restrict__ planes, const long long* __restrict__ info,
                                                         int W, const unsigned long long* __restrict__ B, const float* __restrict__ Bw,
                                                         int Sb, int R, int lds_words, double* __restrict__ out) {
    extern __shared__ unsigned long long As[];
    const int S = static_cast<int>(info[0]);
    const bool neg = info[1] != 0;
    const bool staged = S * W <= lds_words;
    if (staged)
        for (int i = threadIdx.x; i < S * W; i += 256) As[i] = planes[i];
    __syncthreads();
    const int r = blockIdx.x * (256 / kLanes) + static_cast<int>(threadIdx.x) / kLanes;
    const int l = threadIdx.x % kLanes;
    double acc = 0.0;
    if (r < R) {
        const unsigned long long* row = B + static_cast<size_t>(r) * Sb * W;
        for (int w = l; w < W; w += kLanes) {
            for (int j0 = 0; j0 < Sb; j0 += 4) {
                unsigned long long b[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) b[u] = j0 + u < Sb ? row[static_cast<size_t>(j0 + u) * W + w] : 0ULL;
                double part[4];
                auto combine = [&](auto zero) {
                    decltype(zero) t[4] = {zero, zero, zero, zero};
                    for (int i = S - 1; i >= 0; --i) {
                        const unsigned long long a = staged ? As[i * W + w] : planes[static_cast<size_t>(i) * W + w];
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
            }
        }
    }
#pragma unroll
    for (int off = kLanes / 2; off > 0; off >>= 1) acc += __shfl_xor(acc, off, BSI_WAVE);
    if (r < R && l == 0) out[r] = acc;
}

}  // namespace bsi

using namespace bsi;

extern "C" int64_t bsi_hip_scalar_query_max_elems(void) { return kScalarMaxElems; }

extern "C" int bsi_hip_scalar_query_dot(const float* x, int64_t d, int decimal_places, double threshold, uint64_t* workspace,
                                        const uint64_t* B, const float* Bw, int Sb, int64_t R, double* out, int64_t* info,
                                        float* build_ms, float* dot_ms, void* stream) {
    BSI_REQUIRE(d >= 1 && d <= kScalarMaxElems, "d must be in [1, %lld] (got %lld)", static_cast<long long>(kScalarMaxElems),
                static_cast<long long>(d));
    BSI_REQUIRE(R >= 1 && R <= (1 << 24) && Sb >= 1 && Sb <= 64, "bad shape");
    BSI_REQUIRE(x && workspace && B && Bw && out && info && build_ms && dot_ms, "null pointer");
    hipStream_t st = as_stream(stream);
    const int W = static_cast<int>((d + 63) / 64);
    unsigned long long* planes = reinterpret_cast<unsigned long long*>(workspace);
    long long* info_dev = reinterpret_cast<long long*>(workspace + static_cast<size_t>(64) * W);
    hipEvent_t ev[3] = {nullptr, nullptr, nullptr};
    hipError_t err = hipSuccess;
    for (int i = 0; i < 3 && err == hipSuccess; ++i) err = hipEventCreate(&ev[i]);
    if (err == hipSuccess) err = hipEventRecord(ev[0], st);
    if (err == hipSuccess) {
        hipLaunchKernelGGL(scalar_query_kernel, dim3(1), dim3(kScalarBlock), 0, st, x, static_cast<int>(d), W,
                           pow(10.0, static_cast<double>(decimal_places)), threshold, planes, info_dev,
                           reinterpret_cast<long long*>(info));
        err = hipGetLastError();
    }
    if (err == hipSuccess) err = hipEventRecord(ev[1], st);
    if (err == hipSuccess) {
        // the lanes of a row cover its words where they can; 64 KiB of LDS hold 64 slices of 8192 elements
        const int lds_words = 64 * W < 8192 ? 64 * W : 8192;
#define BSI_SCALAR_DOT(L)                                                                                              \
    hipLaunchKernelGGL(scalar_dot_kernel<L>, dim3(static_cast<unsigned>((R + 256 / (L) - 1) / (256 / (L)))), dim3(256),  \
                       static_cast<size_t>(lds_words) * 8, st, planes, info_dev, W,                                     \
                       reinterpret_cast<const unsigned long long*>(B), Bw, Sb, static_cast<int>(R), lds_words, out)
        if (W > 32) BSI_SCALAR_DOT(64);
        else if (W > 16) BSI_SCALAR_DOT(32);
        else BSI_SCALAR_DOT(16);
#undef BSI_SCALAR_DOT
        err = hipGetLastError();
    }
    if (err == hipSuccess) err = hipEventRecord(ev[2], st);
    if (err == hipSuccess) err = hipEventSynchronize(ev[2]);
    if (err == hipSuccess) err = hipEventElapsedTime(build_ms, ev[0], ev[1]);
    if (err == hipSuccess) err = hipEventElapsedTime(dot_ms, ev[1], ev[2]);
    for (hipEvent_t e : ev)
        if (e != nullptr) (void)hipEventDestroy(e);
    if (err != hipSuccess) return fail(BSI_ERR_HIP, "scalar query: %s", hipGetErrorString(err));
    return BSI_OK;
}
