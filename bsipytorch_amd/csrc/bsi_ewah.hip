// EWAH run/literal codec for bit-plane slices (gfx950).
//
// Stream format (one per slice), as in the reference (bsi_ops/csrc/cuda/bsi_cuda_kernels_ewah.cuh:5-33,
// 178-232; bsi_vector_utils.h:74): a sequence of [marker][literal words...], marker =
// run_bit | run_len << 1 | literal_count << 33 (32-bit run length, 31-bit literal count).  A slice
// whose compress flag is 0 is one marker with literal_count = W followed by its W words.
//
// Every kernel here gives one wave to one slice.  Encoding (size pass, emit pass): the wave classifies 64 words at
// a time (literal, zero fill, one fill); a marker starts at word 0 and at every clean word whose predecessor is a
// literal or a clean word of the other kind, so ballots of the three classes give, by population counts, every
// word's place in the stream and every marker's two counts -- no lane walks the slice.  Decoding: the markers of a
// stream form a chain (each one tells where the next sits), which the wave follows through a 64-word window of the
// stream held one word per lane (a lane broadcast per marker instead of a dependent memory load); runs are written
// and literal blocks copied by all lanes together.
#include "bsi_ewah_device.h"

namespace bsi {

constexpr int kEwahBlock = 256;

// one wave per slice
__global__ void slice_popcount_kernel(const unsigned long long* __restrict__ words, int S, int W,
                                      unsigned long long* __restrict__ counts) {
    const int lane = threadIdx.x & (BSI_WAVE - 1);
    const int64_t s = static_cast<int64_t>(blockIdx.x) * (kEwahBlock / BSI_WAVE) + (threadIdx.x >> 6);
    if (s >= S) return;
    const unsigned long long* base = words + static_cast<size_t>(s) * W;
    unsigned long long local = 0ULL;
    for (int w = lane; w < W; w += BSI_WAVE) local += static_cast<unsigned long long>(__popcll(base[w]));
    local = wave_sum_u64(local);
    if (lane == 0) counts[s] = local;
}

__global__ void compress_flags_kernel(const unsigned long long* __restrict__ counts, int S, int W, double threshold,
                                      int* __restrict__ flags) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= S) return;
    flags[s] = compress_flag(counts[s], W, threshold);
}

__global__ void ewah_size_kernel(const unsigned long long* __restrict__ words, int S, int W,
                                 const int* __restrict__ flags, unsigned long long* __restrict__ sizes) {
    const int lane = threadIdx.x & (BSI_WAVE - 1);
    const int64_t s = static_cast<int64_t>(blockIdx.x) * (kEwahBlock / BSI_WAVE) + (threadIdx.x >> 6);
    if (s >= S) return;
    const unsigned long long n = ewah_encode_wave(words + static_cast<size_t>(s) * W, W, flags[s], nullptr, lane);
    if (lane == 0) sizes[s] = n;
}

__global__ void ewah_emit_kernel(const unsigned long long* __restrict__ words, int S, int W,
                                 const int* __restrict__ flags, const unsigned long long* __restrict__ off,
                                 unsigned long long* __restrict__ out, int* __restrict__ out_len) {
    const int lane = threadIdx.x & (BSI_WAVE - 1);
    const int64_t s = static_cast<int64_t>(blockIdx.x) * (kEwahBlock / BSI_WAVE) + (threadIdx.x >> 6);
    if (s >= S) return;
    const unsigned long long n = ewah_encode_wave(words + static_cast<size_t>(s) * W, W, flags[s], out + off[s], lane);
    if (lane == 0) out_len[s] = static_cast<int>(n);
}

// Density flag and stream length of every slice in one pass (the words of a slice are counted, then measured from the
// cache): what slice_popcount, compress_flags and ewah_size give in three launches.  One wave per slice.
__global__ void ewah_measure_kernel(const unsigned long long* __restrict__ words, int S, int W, double threshold,
                                    int* __restrict__ flags, int* __restrict__ lens) {
    const int lane = threadIdx.x & (BSI_WAVE - 1);
    const int64_t s = static_cast<int64_t>(blockIdx.x) * (kEwahBlock / BSI_WAVE) + (threadIdx.x >> 6);
    if (s >= S) return;
    const unsigned long long* base = words + static_cast<size_t>(s) * W;
    unsigned long long count = 0ULL;
    for (int w = lane; w < W; w += BSI_WAVE) count += static_cast<unsigned long long>(__popcll(base[w]));
    const int flag = compress_flag(wave_sum_u64(count), W, threshold);
    const unsigned long long n = flag ? ewah_encode_wave(base, W, 1, nullptr, lane) : static_cast<unsigned long long>(W > 0 ? W + 1 : 0);
    if (lane == 0) {
        flags[s] = flag;
        lens[s] = static_cast<int>(n);
    }
}

// Exclusive sums of the stream lengths, and their total to the host: one workgroup, a run of slices per thread.  The
// total is stored with system scope, so that a host that waits for it need not wait for the kernel to end.
constexpr int kScanBlock = 1024;
__global__ __launch_bounds__(kScanBlock) void ewah_offsets_kernel(const int* __restrict__ lens, int S, long long* __restrict__ off,
                                                                  long long* __restrict__ total_host) {
    __shared__ long long wave_sums[kScanBlock / BSI_WAVE];
    const int tid = threadIdx.x, lane = tid & (BSI_WAVE - 1), wave = tid >> 6;
    const int run = (S + kScanBlock - 1) / kScanBlock;
    const int first = tid * run < S ? tid * run : S, last = first + run < S ? first + run : S;
    long long sum = 0;
    for (int s = first; s < last; ++s) sum += lens[s];
    long long at = sum;  // inclusive over the wave
#pragma unroll
    for (int o = 1; o < BSI_WAVE; o <<= 1) {
        const long long v = __shfl_up(at, o, BSI_WAVE);
        if (lane >= o) at += v;
    }
    if (lane == BSI_WAVE - 1) wave_sums[wave] = at;
    __syncthreads();
    for (int w = 0; w < wave; ++w) at += wave_sums[w];
    if (tid == kScanBlock - 1) __hip_atomic_store(total_host, at, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    at -= sum;
    for (int s = first; s < last; ++s) {
        off[s] = at;
        at += lens[s];
    }
}

// one wave per stream
__global__ void ewah_decompress_batch_kernel(const unsigned long long* __restrict__ comp,
                                             const long long* __restrict__ off, const int* __restrict__ len, int S,
                                             int W, unsigned long long* __restrict__ out) {
    const int lane = threadIdx.x & (BSI_WAVE - 1);
    const int64_t s = static_cast<int64_t>(blockIdx.x) * (kEwahBlock / BSI_WAVE) + (threadIdx.x >> 6);
    if (s >= S) return;
    const long long o = off ? off[s] : 0;
    ewah_expand_wave(comp + o, len[s], W, out + static_cast<size_t>(s) * W, W, lane);
}

__global__ void ewah_decompress_one_kernel(const unsigned long long* __restrict__ in, int in_len, int W,
                                           unsigned long long* __restrict__ out) {
    ewah_expand_wave(in, in_len, W, out, W, static_cast<int>(threadIdx.x));
}

}  // namespace bsi

using namespace bsi;

extern "C" int bsi_hip_slice_popcount_sum(const uint64_t* words, int S, int W, uint64_t* counts, void* stream) {
    BSI_REQUIRE(S >= 0 && W >= 0, "negative size");
    if (S == 0) return BSI_OK;
    BSI_REQUIRE(words && counts, "null pointer");
    const unsigned grid = static_cast<unsigned>((S + 3) / 4);
    launch(slice_popcount_kernel, dim3(grid), dim3(kEwahBlock), 0, as_stream(stream),
                       reinterpret_cast<const unsigned long long*>(words), S, W,
                       reinterpret_cast<unsigned long long*>(counts));
    BSI_LAUNCH_CHECK("slice_popcount_kernel");
    return BSI_OK;
}

extern "C" int bsi_hip_compress_flags_from_density(const uint64_t* counts, int S, int W, double threshold,
                                                   int32_t* flags, void* stream) {
    BSI_REQUIRE(S >= 0 && W >= 0, "negative size");
    if (S == 0) return BSI_OK;
    BSI_REQUIRE(counts && flags, "null pointer");
    launch(compress_flags_kernel, dim3((S + 127) / 128), dim3(128), 0, as_stream(stream),
                       reinterpret_cast<const unsigned long long*>(counts), S, W, threshold, flags);
    BSI_LAUNCH_CHECK("compress_flags_kernel");
    return BSI_OK;
}

extern "C" int bsi_hip_ewah_size(const uint64_t* words, int S, int W, const int32_t* flags, uint64_t* sizes,
                                 void* stream) {
    BSI_REQUIRE(S >= 0 && W >= 0, "negative size");
    if (S == 0) return BSI_OK;
    BSI_REQUIRE(words && flags && sizes, "null pointer");
    launch(ewah_size_kernel, dim3((S + 3) / 4), dim3(kEwahBlock), 0, as_stream(stream),
                       reinterpret_cast<const unsigned long long*>(words), S, W, flags,
                       reinterpret_cast<unsigned long long*>(sizes));
    BSI_LAUNCH_CHECK("ewah_size_kernel");
    return BSI_OK;
}

extern "C" int bsi_hip_ewah_measure(const uint64_t* words, int S, int W, double threshold, int32_t* flags, int32_t* lens,
                                    int64_t* off, int64_t* total_host, void* stream) {
    BSI_REQUIRE(S >= 1 && W >= 0, "bad shape");
    BSI_REQUIRE(words && flags && lens && off && total_host, "null pointer");
    launch(ewah_measure_kernel, dim3((S + 3) / 4), dim3(kEwahBlock), 0, as_stream(stream),
                       reinterpret_cast<const unsigned long long*>(words), S, W, threshold, flags, lens);
    BSI_LAUNCH_CHECK("ewah_measure_kernel");
    launch(ewah_offsets_kernel, dim3(1), dim3(kScanBlock), 0, as_stream(stream), lens, S,
                       reinterpret_cast<long long*>(off), reinterpret_cast<long long*>(total_host));
    BSI_LAUNCH_CHECK("ewah_offsets_kernel");
    return BSI_OK;
}

extern "C" int bsi_hip_ewah_emit(const uint64_t* words, int S, int W, const int32_t* flags, const uint64_t* off,
                                 uint64_t* out, int32_t* out_len, void* stream) {
    BSI_REQUIRE(S >= 0 && W >= 0, "negative size");
    if (S == 0) return BSI_OK;
    BSI_REQUIRE(words && flags && off && out && out_len, "null pointer");
    launch(ewah_emit_kernel, dim3((S + 3) / 4), dim3(kEwahBlock), 0, as_stream(stream),
                       reinterpret_cast<const unsigned long long*>(words), S, W, flags,
                       reinterpret_cast<const unsigned long long*>(off), reinterpret_cast<unsigned long long*>(out),
                       out_len);
    BSI_LAUNCH_CHECK("ewah_emit_kernel");
    return BSI_OK;
}

extern "C" int bsi_hip_ewah_decompress(const uint64_t* in, int in_len, int W, uint64_t* out, void* stream) {
    BSI_REQUIRE(in_len >= 0 && W >= 0, "negative size");
    if (W == 0) return BSI_OK;
    BSI_REQUIRE(out && (in || in_len == 0), "null pointer");
    // one stream = a batch of one: `len` is read from a kernel argument instead of an array
    launch(ewah_decompress_one_kernel, dim3(1), dim3(BSI_WAVE), 0, as_stream(stream),
                       reinterpret_cast<const unsigned long long*>(in), in_len, W,
                       reinterpret_cast<unsigned long long*>(out));
    BSI_LAUNCH_CHECK("ewah_decompress_one_kernel");
    return BSI_OK;
}

extern "C" int bsi_hip_ewah_decompress_batch(const uint64_t* comp, const int64_t* off, const int32_t* len, int S,
                                             int W, uint64_t* out, void* stream) {
    BSI_REQUIRE(S >= 0 && W >= 0, "negative size");
    if (S == 0 || W == 0) return BSI_OK;
    BSI_REQUIRE(comp && off && len && out, "null pointer");
    launch(ewah_decompress_batch_kernel, dim3((S + 3) / 4), dim3(kEwahBlock), 0, as_stream(stream),
                       reinterpret_cast<const unsigned long long*>(comp), reinterpret_cast<const long long*>(off), len,
                       S, W, reinterpret_cast<unsigned long long*>(out));
    BSI_LAUNCH_CHECK("ewah_decompress_batch_kernel");
    return BSI_OK;
}
