// The dot for a few query rows (decode steps): kernels that stream the packed key planes once -- on a built int8
// query image, with the query build inside, or with queries handed over as EWAH streams -- and the stream -> int8
// image pass for larger batches of EWAH queries.  Shapes in the comments are rows x width x keys.
#include "bsi_dot_internal.h"
#include "bsi_coop_build.h"
#include <type_traits>

namespace bsi {

// ------------------------------------------------------------------ MFMA core, few query rows
//
// Decode-like shapes (a handful of query rows against a large key matrix) are bound by reading the
// packed key planes once.  One workgroup owns one 16-key tile of the tiled layout over all chunks
// and up to 16 * NT query rows; its waves take the chunks round-robin.  A lane loads the six plane
// words of (key row lane % 16, 64-bit word lane / 16), transposes them in registers into the four
// 16-byte MFMA operands of that row (no LDS staging: with a k permutation shared by both operands
// any assignment of chunk elements to MFMA k-slots gives the same integer), loads the matching 64
// int8 query bytes from L2, and issues 4 MFMAs per query tile.  The int32 results go to LDS
// indexed by chunk; after a workgroup barrier 256 * NT lanes run the fp32 chain of their (query,
// key) pair over the chunks in order, so the result is bit-identical to a sequential pass
// whatever the number of waves.  Problems with more chunks than LDS slots run in several passes.

constexpr int kStreamLdsInts = 16384;  // at most 64 KiB of chunk accumulators per pass
constexpr int kStreamLds = kStreamLdsInts * 4 + 4096 + 16 * 2048;  // with their scales and 16 waves' query rows

// kBuild: the queries are quantised by this launch (bsi_coop_build.h; 1: a chunk a wave at a time, 2: a row); A8 and qscale are
// not looked at.  The copy lies in the order of the operand loads (coop_image_at: up to 1 KiB in one run a load, where rows one
// after the other are 32 lines a load and the loads of 32 rows take longer than the key planes they are for), and a wave takes a
// chunk's scales with its operands and leaves them in LDS, so that the chain asks memory for nothing.  us a layer, rows and the chain's own loads before, then now:
// 16 x 4096 x 4096 bf16 8.7, 7.85; 32 x 4096 x 4096 11.05, 8.95; 32 x 8192 x 4096 f16 16.5, 12.4; 16 x 8192 x 4096 12.1, 10.5;
// 24 x 2048 x 2048 f32 6.95, 6.25; 8 x 4096 x 4096 7.8, 7.6.  Only those instances
// take the build's description: with it the workgroup's size, which lies behind the arguments, is in another cache line of
// them, and its fetch holds up every wave's first key load.  us, with and without: 16 x 4096 x 16384 12.3, 11.8; 16 x 4096 x
// 4096 5.25, 5.09; 1 x 4096 x 16384 10.5, 10.2; 1 x 16384 x 4096 11.1, 10.9 (1 x 4096 x 4096 4.06, 4.11).
//
// Without kBuild the image has its rows one after the other.  An operand's lanes want 64 bytes of each of 16 rows, and loads of
// such pieces run at half the rate of whole lines (a chunk is 3 KiB of a key tile's planes and 4 KiB of 16 query rows, which then
// take as long as 8); so a load takes 128 bytes of 8 rows, and the wave turns them round through 2 KiB of LDS, in which its sums lie afterwards.  The scales
// go with them, as above.  us a dot, operands straight from memory, then so: 16 x 16384 x 4096 14.7, 12.2; 16 x 8192 x 8192 13.9,
// 11.9; 24 x 8192 x 8192 18.7, 14.8; 32 x 4096 x 4096 7.6, 6.1; 16 x 8192 x 32768 44.8, 41.0; 8 x 16384 x 4096 12.6, 11.9;
// 1 x 4096 x 32768 21.6, 21.5; 8 x 8192 x 16384 21.5, 21.5.  All 4 KiB of a chunk at once, in LDS of its own: 12.0 for the first,
// but 22.5 for the last (a workgroup less on a CU).
template <int NT, int KT, bool kInts, int kBuild>
__global__ __launch_bounds__(1024) void dot_mfma_stream_kernel(
    const int8_t* A8, const float* qscale, int qscale_stride,
    const unsigned long long* __restrict__ B64,  // tiled key planes, Sb = 6
    const float* __restrict__ Bw, int chunks, int pass_chunks, int64_t R, int64_t Q, int down_shift, float scale_inv,
    int64_t R_total, float* __restrict__ out, int* __restrict__ chunk_ints, const float* __restrict__ bias, int out_dtype,
    std::conditional_t<kBuild != 0, CoopBuild, int> coop) {
    // [pass_chunks][KT][NT][16 queries][16 keys], then the chunks' scales, [pass_chunks][NT][16 queries]; without kBuild a chunk's
    // query rows are turned round where its sums will lie, or, if those have no 2 KiB, in 2 KiB a wave behind all that
    extern __shared__ __attribute__((aligned(16))) int ints[];
    constexpr int kSlot = KT * NT * 256;
    float* const chunk_scales = reinterpret_cast<float*>(ints + static_cast<size_t>(pass_chunks) * kSlot);

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nwaves = static_cast<int>(blockDim.x >> 6);
    const int ln = lane & 15, lg = lane >> 4;
    const int64_t ntiles = (R + 15) / 16;
    const int64_t tile0 = static_cast<int64_t>(blockIdx.x) * KT;
    const int64_t q0 = static_cast<int64_t>(blockIdx.y) * (16 * NT);
    const size_t ktile = static_cast<size_t>(chunks) * (6 * 64);  // words per key tile
    const unsigned long long* ksrc[KT];
#pragma unroll
    for (int k = 0; k < KT; ++k) {
        const int64_t t = (tile0 + k < ntiles) ? tile0 + k : ntiles - 1;  // clamped: its outputs are never stored
        ksrc[k] = B64 + static_cast<size_t>(t) * ktile + lane;
    }
    const size_t arow = static_cast<size_t>(chunks) * 256;
    // without kBuild: rows past the batch read 0; kMfmaMaxChunks keeps 32 rows of an image below 2^31 bytes
    [[maybe_unused]] const int64_t rows_here = Q - q0 < NT * 16 ? Q - q0 : NT * 16;
    [[maybe_unused]] const bsi_rsrc qrs = make_rsrc(A8 + static_cast<size_t>(q0) * arow, static_cast<size_t>(rows_here) * arow);
    [[maybe_unused]] const bsi_rsrc srs = make_rsrc(qscale + q0 * qscale_stride, static_cast<size_t>(rows_here) * qscale_stride * 4);
    [[maybe_unused]] v4i* const turn_here = reinterpret_cast<v4i*>(chunk_scales + static_cast<size_t>(pass_chunks) * NT * 16) + wave * 128;
    uint2 kc[KT][6];
    auto load_keys = [&](int c) {
#pragma unroll
        for (int k = 0; k < KT; ++k)
#pragma unroll
            for (int j = 0; j < 6; ++j) {
                const unsigned long long w = ksrc[k][(static_cast<size_t>(c) * 6 + j) * 64];
                kc[k][j] = make_uint2(static_cast<uint32_t>(w), static_cast<uint32_t>(w >> 32));
            }
    };
    // Workgroups beyond the tiles, there for the build (coop_groups), go on with the last tile and store nothing: a branch past the rest
    // costs the others 0.2 us (16 x 4096 x 4096 7.8 -> 8.0).
    if constexpr (kBuild)
        coop_build<true, kBuild == 2>(coop, blockIdx.x, reinterpret_cast<unsigned*>(ints), A8, qscale, [&] { load_keys(wave < pass_chunks ? wave : pass_chunks - 1); });

    // the chain lanes: tid <-> (key tile, query tile, query, key), keys fastest so output stores are contiguous
    float accf = 0.0f;
    const bool chain = tid < kSlot;
    const int ck = tid / (NT * 256), ct = (tid >> 8) % NT, cn = (tid >> 4) & 15, ckey = tid & 15;
    const int64_t cq = q0 + ct * 16 + cn, cr = (tile0 + ck) * 16 + ckey;
    const bool cvalid = chain && cq < Q && cr < R;
    const float down = __uint_as_float(static_cast<uint32_t>(127 - down_shift) << 23);
    const EpilogueOperands eo = load_epilogue_operands(Bw, bias, R, cvalid, cr);

    // passes but the last are whole rounds of the waves, so that a wave's next chunk is nwaves further on across them too and its
    // planes are on their way while the chain runs
    if (!kBuild) load_keys(wave < chunks ? wave : chunks - 1);
    for (int p0 = 0; p0 < chunks; p0 += pass_chunks) {
        const int pend = (p0 + pass_chunks < chunks) ? p0 + pass_chunks : chunks;
        for (int c = p0 + wave; c < pend; c += nwaves) {
            // query operands of this chunk (L2 resident), then the key planes of the wave's next chunk
            v4i qb[NT][4];
            float qs[NT];
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                if constexpr (kBuild) {
                    qs[t] = 0.0f;
                    if (q0 + t * 16 + ln < Q) {
                        const int rows = Q - t * 16 < 16 ? static_cast<int>(Q) - t * 16 : 16;  // coop_image_at's order
                        const v4i* src = reinterpret_cast<const v4i*>(A8 + static_cast<size_t>(t) * 16 * arow + ((c * 16 + lg) * rows + ln) * 16);
                        qs[t] = qscale[coop.by_row ? t * 16 + ln : t * 16 * chunks + c * rows + ln];
#pragma unroll
                        for (int m = 0; m < 4; ++m) qb[t][m] = src[m * 4 * rows];
                    } else {
#pragma unroll
                        for (int m = 0; m < 4; ++m) qb[t][m] = (v4i){0, 0, 0, 0};
                    }
                } else {
                    const int uc = __builtin_amdgcn_readfirstlane(c);
                    qs[t] = __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(srs, (t * 16 + ln) * qscale_stride * 4,
                                                                                qscale_stride == 1 ? 0 : uc * 4, 0));
#pragma unroll
                    for (int m = 0; m < 4; ++m)  // 128 bytes of 8 rows
                        qb[t][m] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(
                            qrs, (t * 16 + (m & 1) * 8 + (lane >> 3)) * chunks * 256 + (m >> 1) * 128 + (lane & 7) * 16, uc * 256, 0));
                }
            }
            uint2 kn[KT][6];
            const int cnext = c + nwaves;
            if (cnext < chunks) {
#pragma unroll
                for (int k = 0; k < KT; ++k)
#pragma unroll
                    for (int j = 0; j < 6; ++j) {
                        const unsigned long long w = ksrc[k][(static_cast<size_t>(cnext) * 6 + j) * 64];
                        kn[k][j] = make_uint2(static_cast<uint32_t>(w), static_cast<uint32_t>(w >> 32));
                    }
            }
            if constexpr (!kBuild) {
                // half a chunk of 16 rows at a time; 16-byte column x of row r lies at x ^ (r & 7): conflict-free both ways.  A
                // wave's LDS instructions are done in order.
                v4i* const turn = kSlot >= 512 ? reinterpret_cast<v4i*>(ints + (c - p0) * kSlot) : turn_here;
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const v4i loaded[4] = {qb[t][0], qb[t][1], qb[t][2], qb[t][3]};
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        turn[lane ^ (lane >> 3)] = loaded[h * 2];
                        turn[64 + (lane ^ (lane >> 3))] = loaded[h * 2 + 1];
                        __builtin_amdgcn_wave_barrier();
                        if ((lg >> 1) == h) {
#pragma unroll
                            for (int m = 0; m < 4; ++m) qb[t][m] = turn[ln * 8 + (((lg & 1) * 4 + m) ^ (ln & 7))];
                        }
                        __builtin_amdgcn_wave_barrier();
                    }
                }
            }
#pragma unroll
            for (int k = 0; k < KT; ++k) {
                uint32_t lo[8], hi[8];
                transpose_6planes(kc[k][0].x, kc[k][1].x, kc[k][2].x, kc[k][3].x, kc[k][4].x, kc[k][5].x, lo);
                transpose_6planes(kc[k][0].y, kc[k][1].y, kc[k][2].y, kc[k][3].y, kc[k][4].y, kc[k][5].y, hi);
                v4i ka[4];
                ka[0] = (v4i){static_cast<int>(lo[0]), static_cast<int>(lo[1]), static_cast<int>(lo[2]), static_cast<int>(lo[3])};
                ka[1] = (v4i){static_cast<int>(lo[4]), static_cast<int>(lo[5]), static_cast<int>(lo[6]), static_cast<int>(lo[7])};
                ka[2] = (v4i){static_cast<int>(hi[0]), static_cast<int>(hi[1]), static_cast<int>(hi[2]), static_cast<int>(hi[3])};
                ka[3] = (v4i){static_cast<int>(hi[4]), static_cast<int>(hi[5]), static_cast<int>(hi[6]), static_cast<int>(hi[7])};
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    v4i acc = {0, 0, 0, 0};
#pragma unroll
                    for (int m = 0; m < 4; ++m) acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(ka[m], qb[t][m], acc, 0, 0, 0);
                    // the lane holds keys 4*lg .. 4*lg+3 of query ln
                    *reinterpret_cast<v4i*>(&ints[(c - p0) * kSlot + (k * NT + t) * 256 + ln * 16 + lg * 4]) = acc;
                }
            }
            if (lg == 0) {
#pragma unroll
                for (int t = 0; t < NT; ++t) chunk_scales[((c - p0) * NT + t) * 16 + ln] = qs[t];
            }
            if (cnext < chunks) {
#pragma unroll
                for (int k = 0; k < KT; ++k)
#pragma unroll
                    for (int j = 0; j < 6; ++j) kc[k][j] = kn[k][j];
            }
        }
        __syncthreads();
        if (cvalid) {
            accf = chain_chunks(accf, p0, pend, down, [&](int cc) { return ints[(cc - p0) * kSlot + tid]; },
                                [&](int cc) { return chunk_scales[((cc - p0) * NT + ct) * 16 + cn]; });
            if (kInts)
                for (int cc = p0; cc < pend; ++cc)
                    chunk_ints[(cq * R + cr) * chunks + cc] = ints[(cc - p0) * kSlot + tid] >> down_shift;
        }
        if (pend < chunks) __syncthreads();
    }
    if (cvalid)
        store_output(out, static_cast<size_t>(cq) * R_total + cr, (accf * eo.bw) * scale_inv, bias != nullptr, eo.bias, out_dtype);
}

// The few-rows kernel with the query build inside (at most kFusedMaxQ rows: a decode step).  Every workgroup first
// issues the loads of its first key planes, then quantises the activations itself while those are in flight: the
// (chunk, row) items go round-robin over the waves, each one the builder's per-chunk routine -- round half away of
// x * 10^dec, the chunk's shift from its largest magnitude, rounded shift and clamp -- and leave the int8 MFMA
// operand and the chunk scale in LDS.  After a barrier the kernel is the few-rows kernel above with its query
// operand in LDS.  Every workgroup repeats that small amount of arithmetic (a few hundred VALU cycles per wave
// against microseconds of key traffic), and a BSI-linear layer becomes ONE launch instead of a build and a dot.
// Same integers, scales and fp32 chain as bsi_hip_build_fixed + bsi_hip_dot, so the same bits.
constexpr int kFusedMaxQ = 4;
constexpr size_t kFusedQueryLdsBytes = 96 * 1024;  // int8 image + chunk scales of all rows: chunks * Q * 260 bytes

template <typename T, int KT, int NI, bool kVec>
__global__ __launch_bounds__(1024) void dot_mfma_stream_fused_kernel(
    const T* __restrict__ x, int64_t d, double dec_scale, int narrow, int slices,
    const unsigned long long* __restrict__ B64,  // tiled key planes, Sb = 6
    const float* __restrict__ Bw, int chunks, int pass_chunks, int64_t R, int Q, float scale_inv, int64_t R_total,
    float* __restrict__ out, const float* __restrict__ bias, int out_dtype) {
    // [pass_chunks][KT][16 queries][16 keys] ints | [chunks][Q][256] image bytes | [chunks][Q] scales
    extern __shared__ __attribute__((aligned(16))) int ints[];
    constexpr int kSlot = KT * 256;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nwaves = static_cast<int>(blockDim.x >> 6);
    const int ln = lane & 15, lg = lane >> 4;
    unsigned char* const qimg = reinterpret_cast<unsigned char*>(ints + static_cast<size_t>(pass_chunks) * kSlot);
    float* const qsc = reinterpret_cast<float*>(qimg + static_cast<size_t>(chunks) * Q * 256);
    const int64_t ntiles = (R + 15) / 16;
    const int64_t tile0 = static_cast<int64_t>(blockIdx.x) * KT;
    const size_t ktile = static_cast<size_t>(chunks) * (6 * 64);  // words per key tile
    const unsigned long long* ksrc[KT];
#pragma unroll
    for (int k = 0; k < KT; ++k) {
        const int64_t t = (tile0 + k < ntiles) ? tile0 + k : ntiles - 1;  // clamped: its outputs are never stored
        ksrc[k] = B64 + static_cast<size_t>(t) * ktile + lane;
    }
    const int down_shift = 16 - slices - 6;

    // the chain lanes: tid <-> (key tile, query, key), keys fastest so output stores are contiguous
    float accf = 0.0f;
    const int ck = tid >> 8, cn = (tid >> 4) & 15, ckey = tid & 15;
    const int64_t cr = (tile0 + ck) * 16 + ckey;
    const bool cvalid = tid < kSlot && cn < Q && cr < R;
    const float down = __uint_as_float(static_cast<uint32_t>(127 - down_shift) << 23);

    // The wave's share of the query build: (chunk, row) items wave, wave + nwaves, ...  The loads of a CU return in
    // order, so the activations are requested BEFORE the first key planes (they would otherwise wait behind that
    // traffic, one round trip per item) and all at once: up to kFusedItems items per wave sit in registers while
    // the key loads are issued, then they are quantised under the latency of those.
    constexpr int kFusedItems = NI;  // 1, 2 or (one key tile only) 4: what the registers hold beside the key planes
    const int items = chunks * Q;
    // Buffer loads, one descriptor per row: past the row's end they return 0 without a branch (with loads in
    // conditional blocks the compiler waits for every outstanding load, the key planes included, before a use).
    const ChunkLane cl = chunk_lane(lane);
    const QuantRange range = quant_range(slices);
    const float scale = static_cast<float>(dec_scale);
    auto load_item = [&](int item, float (&dst)[4]) {
        const int ic = item / Q, iq = item - ic * Q;
        load_chunk_quad<T, kVec>(x + static_cast<int64_t>(iq) * d, d, ic, cl, dst);
    };
    // One item: 256 image bytes and one scale into LDS.  narrow: 10^dec is an integer of at most 127 (quantise_quad's range).
    auto quantize = [&](int item, const float (&xv)[4]) {
        const unsigned mx = wave_max_u32(quad_max_bits(xv));
        int shift;
        uint32_t bytes;
        if (narrow && mx < kQuantWideBits) {
            shift = quant_shift(mx, scale, slices);
            bytes = quantise_quad<T>(xv, scale, shift, range);
        } else {
            shift = compute_shift(wave_max_u64(quad_max_wide(xv, dec_scale)), 0.0, 1, slices, 0.0f);
            bytes = quantise_quad_wide(xv, dec_scale, shift, slices);
        }
        reinterpret_cast<uint32_t*>(qimg)[item * 64 + lane] = chunk_image_dword(bytes, cl);
        if (lane == 0) qsc[item] = static_cast<float>(1ULL << shift);
    };
    float xr[kFusedItems][4];
#pragma unroll
    for (int i = 0; i < kFusedItems; ++i) {
        const int item = wave + i * nwaves;
        load_item(item < items ? item : items - 1, xr[i]);
    }

    uint2 kc[KT][6];
    auto load_keys = [&](int chunk, uint2 (&dst)[KT][6]) {
#pragma unroll
        for (int k = 0; k < KT; ++k)
#pragma unroll
            for (int j = 0; j < 6; ++j) {
                const unsigned long long w = ksrc[k][(static_cast<size_t>(chunk) * 6 + j) * 64];
                dst[k][j] = make_uint2(static_cast<uint32_t>(w), static_cast<uint32_t>(w >> 32));
            }
    };
    // the first pass's first chunk; a wave without one loads the last chunk's planes for nothing, because a branch
    // here would make the compiler's load counting assume the worst and wait for these loads in the query build
    load_keys(wave < pass_chunks ? wave : pass_chunks - 1, kc);
    const EpilogueOperands eo = load_epilogue_operands(Bw, bias, R, cvalid, cr);
    __builtin_amdgcn_sched_barrier(0);
    {
#pragma unroll
        for (int i = 0; i < kFusedItems; ++i) {
            // no branch here either (the compiler would sink the item's loads into it, behind the key loads): a wave
            // with fewer items repeats the last one, and writes the bytes its owner writes
            const int item = wave + i * nwaves;
            quantize(item < items ? item : items - 1, xr[i]);
            __builtin_amdgcn_sched_barrier(0);  // one item at a time: interleaving them costs registers, gains nothing
        }
        // longer rows: the rest one item at a time (each waits for its own loads)
#pragma unroll 1
        for (int item = wave + kFusedItems * nwaves; item < items; item += nwaves) {
            float xa[4];
            load_item(item, xa);
            quantize(item, xa);
        }
        __syncthreads();
    }

    for (int p0 = 0; p0 < chunks; p0 += pass_chunks) {
        const int pend = (p0 + pass_chunks < chunks) ? p0 + pass_chunks : chunks;
        int c = p0 + wave;
        if (p0 > 0 && c < pend) load_keys(c, kc);
        for (; c < pend; c += nwaves) {
            // query operand of this chunk from LDS, then the key planes of the wave's next chunk
            v4i qb[4];
            if (ln < Q) {
                const v4i* src = reinterpret_cast<const v4i*>(qimg + (static_cast<size_t>(c) * Q + ln) * 256 + lg * 64);
#pragma unroll
                for (int m = 0; m < 4; ++m) qb[m] = src[m];
            } else {
#pragma unroll
                for (int m = 0; m < 4; ++m) qb[m] = (v4i){0, 0, 0, 0};
            }
            uint2 kn[KT][6];
            const int cnext = c + nwaves;
            if (cnext < pend) {
#pragma unroll
                for (int k = 0; k < KT; ++k)
#pragma unroll
                    for (int j = 0; j < 6; ++j) {
                        const unsigned long long w = ksrc[k][(static_cast<size_t>(cnext) * 6 + j) * 64];
                        kn[k][j] = make_uint2(static_cast<uint32_t>(w), static_cast<uint32_t>(w >> 32));
                    }
            }
#pragma unroll
            for (int k = 0; k < KT; ++k) {
                uint32_t lo[8], hi[8];
                transpose_6planes(kc[k][0].x, kc[k][1].x, kc[k][2].x, kc[k][3].x, kc[k][4].x, kc[k][5].x, lo);
                transpose_6planes(kc[k][0].y, kc[k][1].y, kc[k][2].y, kc[k][3].y, kc[k][4].y, kc[k][5].y, hi);
                v4i ka[4];
                ka[0] = (v4i){static_cast<int>(lo[0]), static_cast<int>(lo[1]), static_cast<int>(lo[2]), static_cast<int>(lo[3])};
                ka[1] = (v4i){static_cast<int>(lo[4]), static_cast<int>(lo[5]), static_cast<int>(lo[6]), static_cast<int>(lo[7])};
                ka[2] = (v4i){static_cast<int>(hi[0]), static_cast<int>(hi[1]), static_cast<int>(hi[2]), static_cast<int>(hi[3])};
                ka[3] = (v4i){static_cast<int>(hi[4]), static_cast<int>(hi[5]), static_cast<int>(hi[6]), static_cast<int>(hi[7])};
                v4i acc = {0, 0, 0, 0};
#pragma unroll
                for (int m = 0; m < 4; ++m) acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(ka[m], qb[m], acc, 0, 0, 0);
                // the lane holds keys 4*lg .. 4*lg+3 of query ln
                *reinterpret_cast<v4i*>(&ints[(c - p0) * kSlot + k * 256 + ln * 16 + lg * 4]) = acc;
            }
            if (cnext < pend) {
#pragma unroll
                for (int k = 0; k < KT; ++k)
#pragma unroll
                    for (int j = 0; j < 6; ++j) kc[k][j] = kn[k][j];
            }
        }
        __syncthreads();
        if (cvalid) {
            accf = chain_chunks(accf, p0, pend, down, [&](int cc) { return ints[(cc - p0) * kSlot + tid]; },
                                [&](int cc) { return qsc[cc * Q + cn]; });
        }
        if (pend < chunks) __syncthreads();
    }
    if (cvalid)
        store_output(out, static_cast<size_t>(cn) * R_total + cr, (accf * eo.bw) * scale_inv, bias != nullptr, eo.bias, out_dtype);
}

// ------------------------------------------------------------------ EWAH-compressed queries, decode inline
//
// The hybrid query form keeps each of a query's Sa slices as an EWAH stream ([marker][literals...],
// marker = run_bit | run_len << 1 | literal_count << 33; bsi_cuda_kernels_ewah.cuh:5-33 is the
// decoder this follows, including its bounds: output clipped at W words, input at the stream's
// length, the rest zero).  This kernel is the few-rows kernel for up to 16 such queries per workgroup
// (stream q * Sa + s is slice s of query q) with the decode folded into its load stage: every workgroup
// first expands the streams into bit planes in LDS (a wave per stream: ewah_expand_wave), then
// recombines the planes of each chunk into the int8 MFMA operand in registers, exactly as it does for
// the key planes it streams from HBM.  A slice whose stream says "all zero" (one marker, a zero run
// over the whole slice: the sign plane of ReLU'd activations, the high planes of small values) is not
// expanded at all: its plane reads as zero without touching LDS.
constexpr int kEwahQueriesPerGroup = 16;
__host__ __device__ inline int ewah_stream_stride(int wpad) { return wpad + 1; }  // odd stride: queries spread over the banks
// bytes of the plane region of `group` queries (a multiple of 16: the accumulators behind it are stored 16 bytes at a time)
__host__ __device__ inline size_t ewah_plane_region(int group, int Sa, int wpad) {
    return (static_cast<size_t>(group) * Sa * ewah_stream_stride(wpad) * 8 + 15) & ~static_cast<size_t>(15);
}

// Whether the stream is the encoder's form of an all-zero slice of W words (every lane gets the answer).
__device__ __forceinline__ bool ewah_stream_is_zero(const unsigned long long* __restrict__ in, int in_len, int W) {
    if (in_len == 0) return true;
    if (in_len != 1) return false;
    const unsigned long long m = in[0];
    return (m & 1ULL) == 0ULL && ((m >> 1) & 0xFFFFFFFFULL) >= static_cast<unsigned long long>(W);
}

template <bool kInts>
__global__ __launch_bounds__(1024) void dot_mfma_stream_ewah_kernel(
    const unsigned long long* __restrict__ comp, const long long* __restrict__ comp_off,
    const int* __restrict__ comp_len, int Sa, int W64, const float* __restrict__ qscale, int qscale_stride,
    const unsigned long long* __restrict__ B64,  // tiled key planes, Sb = 6
    const float* __restrict__ Bw, int chunks, int pass_chunks, int64_t R, int64_t Q, int group, int down_shift,
    float scale_inv, int64_t R_total, const float* __restrict__ bias, float* __restrict__ out,
    int* __restrict__ chunk_ints) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    // group = queries per workgroup (min(Q, 16)); LDS: [group][Sa] streams of ewah_stream_stride(4 * chunks) plane
    // words, one presence byte per stream (128 bytes), then the chunk accumulators
    const int wpad = chunks * 4, sstride = ewah_stream_stride(wpad);
    const int64_t q0 = static_cast<int64_t>(blockIdx.y) * kEwahQueriesPerGroup;
    const int nq = static_cast<int>((Q - q0) < kEwahQueriesPerGroup ? (Q - q0) : kEwahQueriesPerGroup);
    const int nstreams = nq * Sa;
    unsigned long long* planes = reinterpret_cast<unsigned long long*>(smem);
    unsigned char* present = smem + ewah_plane_region(group, Sa, wpad);
    int* ints = reinterpret_cast<int*>(present + 128);

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nwaves = static_cast<int>(blockDim.x >> 6);
    const int ln = lane & 15, lg = lane >> 4;
    const int64_t tile = blockIdx.x;
    const unsigned long long* ksrc = B64 + static_cast<size_t>(tile) * chunks * (6 * 64) + lane;

    // ---- inline EWAH decode: the group's streams round-robin over the waves.  Three kinds of stream: all zero
    // (nothing to do), verbatim (one marker followed by the W64 words of the slice: the words are read where they
    // lie, straight from the stream, when their chunk comes up), anything else (expanded into LDS planes now).
    for (int s = wave; s < nstreams; s += nwaves) {
        const unsigned long long* in = comp + comp_off[q0 * Sa + s];
        const int in_len = comp_len[q0 * Sa + s];
        const bool zero = ewah_stream_is_zero(in, in_len, W64);
        const bool verbatim = !zero && in_len == W64 + 1 && in[0] == (static_cast<unsigned long long>(W64) << 33);
        if (lane == 0) present[s] = zero ? 0 : (verbatim ? 2 : 1);
        if (!zero && !verbatim) ewah_expand_wave(in, in_len, W64, planes + static_cast<size_t>(s) * sstride, wpad, lane);
    }
    __syncthreads();

    const bool chain = tid < 256;
    const int ckey = tid & 15, cn = (tid >> 4) & 15;
    const int64_t cr = tile * 16 + ckey;
    const bool cvalid = chain && cn < nq && cr < R;
    const float down = __uint_as_float(static_cast<uint32_t>(127 - down_shift) << 23);
    const int sstep = (qscale_stride == 1) ? 0 : 1;
    const float* myscale = qscale + (q0 + (cn < nq ? cn : 0)) * qscale_stride;
    float accf = 0.0f;
    // the planes of the lane's query (row t of the 8 x 8 transposes): expanded in LDS (have), verbatim in the stream (verb)
    unsigned have = 0, verb = 0;
    const unsigned long long* vptr[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        const int j = t - (8 - Sa);
        vptr[t] = comp;
        if (ln < nq && j >= 0) {
            const int cls = present[ln * Sa + j];
            if (cls == 1) have |= 1u << t;
            if (cls == 2) {
                verb |= 1u << t;
                vptr[t] = comp + comp_off[(q0 + ln) * Sa + j] + 1;  // past the marker
            }
        }
    }
    const unsigned long long* myplanes = planes + static_cast<size_t>(ln < nq ? ln : 0) * Sa * sstride;

    for (int p0 = 0; p0 < chunks; p0 += pass_chunks) {
        const int pend = (p0 + pass_chunks < chunks) ? p0 + pass_chunks : chunks;
        for (int c = p0 + wave; c < pend; c += nwaves) {
            uint2 kc[6];
#pragma unroll
            for (int j = 0; j < 6; ++j) {
                const unsigned long long w = ksrc[(static_cast<size_t>(c) * 6 + j) * 64];
                kc[j] = make_uint2(static_cast<uint32_t>(w), static_cast<uint32_t>(w >> 32));
            }
            // the query operand of this chunk from the decoded planes: MFMA column ln is query q0 + ln
            uint32_t qlo[8], qhi[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                const int j = t - (8 - Sa);
                unsigned long long w = 0ULL;
                if ((verb >> t) & 1u) w = (c * 4 + lg < W64) ? vptr[t][c * 4 + lg] : 0ULL;
                else if ((have >> t) & 1u) w = myplanes[static_cast<size_t>(j) * sstride + c * 4 + lg];
                qlo[t] = static_cast<uint32_t>(w);
                qhi[t] = static_cast<uint32_t>(w >> 32);
            }
            transpose8x8(qlo);
            transpose8x8(qhi);
            v4i qb[4];
            qb[0] = (v4i){static_cast<int>(qlo[0]), static_cast<int>(qlo[1]), static_cast<int>(qlo[2]), static_cast<int>(qlo[3])};
            qb[1] = (v4i){static_cast<int>(qlo[4]), static_cast<int>(qlo[5]), static_cast<int>(qlo[6]), static_cast<int>(qlo[7])};
            qb[2] = (v4i){static_cast<int>(qhi[0]), static_cast<int>(qhi[1]), static_cast<int>(qhi[2]), static_cast<int>(qhi[3])};
            qb[3] = (v4i){static_cast<int>(qhi[4]), static_cast<int>(qhi[5]), static_cast<int>(qhi[6]), static_cast<int>(qhi[7])};
            uint32_t lo[8], hi[8];
            transpose_6planes(kc[0].x, kc[1].x, kc[2].x, kc[3].x, kc[4].x, kc[5].x, lo);
            transpose_6planes(kc[0].y, kc[1].y, kc[2].y, kc[3].y, kc[4].y, kc[5].y, hi);
            v4i ka[4];
            ka[0] = (v4i){static_cast<int>(lo[0]), static_cast<int>(lo[1]), static_cast<int>(lo[2]), static_cast<int>(lo[3])};
            ka[1] = (v4i){static_cast<int>(lo[4]), static_cast<int>(lo[5]), static_cast<int>(lo[6]), static_cast<int>(lo[7])};
            ka[2] = (v4i){static_cast<int>(hi[0]), static_cast<int>(hi[1]), static_cast<int>(hi[2]), static_cast<int>(hi[3])};
            ka[3] = (v4i){static_cast<int>(hi[4]), static_cast<int>(hi[5]), static_cast<int>(hi[6]), static_cast<int>(hi[7])};
            v4i acc = {0, 0, 0, 0};
#pragma unroll
            for (int m = 0; m < 4; ++m) acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(ka[m], qb[m], acc, 0, 0, 0);
            *reinterpret_cast<v4i*>(&ints[(c - p0) * 256 + ln * 16 + lg * 4]) = acc;
        }
        __syncthreads();
        if (cvalid) {
            accf = chain_chunks(accf, p0, pend, down, [&](int cc) { return ints[(cc - p0) * 256 + cn * 16 + ckey]; },
                                [&](int cc) { return myscale[cc * sstep]; });
            if (kInts)
                for (int cc = p0; cc < pend; ++cc)
                    chunk_ints[((q0 + cn) * R + cr) * chunks + cc] = ints[(cc - p0) * 256 + cn * 16 + ckey] >> down_shift;
        }
        if (pend < chunks) __syncthreads();
    }
    if (cvalid) {
        float v = (accf * Bw[cr * 6]) * scale_inv;
        if (bias != nullptr) v = v + bias[cr];
        out[(q0 + cn) * R_total + cr] = v;
    }
}

// EWAH streams of a whole query batch -> the int8 query image the compute-bound dot contracts (value << (8 - Sa),
// in-chunk byte order of planes_to_int8_kernel): one workgroup per query row expands the row's Sa streams into LDS
// (a wave per stream, all-zero slices skipped) and recombines them 32 elements per thread.  The verbatim planes
// never exist in memory.
constexpr int kEwahToInt8Block = 512;  // 8 waves: the (at most 8) streams of a row decode side by side
__global__ __launch_bounds__(kEwahToInt8Block) void ewah_streams_to_int8_kernel(const unsigned long long* __restrict__ comp,
                                                                    const long long* __restrict__ comp_off,
                                                                    const int* __restrict__ comp_len, int Sa, int W64,
                                                                    int chunks, uint32_t* __restrict__ out32) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int wpad = chunks * 4;
    unsigned long long* planes = reinterpret_cast<unsigned long long*>(smem);  // [Sa][wpad]
    unsigned char* present = smem + static_cast<size_t>(Sa) * wpad * 8;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t row = blockIdx.x;
    for (int s = wave; s < Sa; s += kEwahToInt8Block / BSI_WAVE) {
        const unsigned long long* in = comp + comp_off[row * Sa + s];
        const int in_len = comp_len[row * Sa + s];
        const bool zero = ewah_stream_is_zero(in, in_len, W64);
        if (lane == 0) present[s] = zero ? 0 : 1;
        if (!zero) ewah_expand_wave(in, in_len, W64, planes + static_cast<size_t>(s) * wpad, wpad, lane);
    }
    __syncthreads();
    const uint32_t* planes32 = reinterpret_cast<const uint32_t*>(planes);
    const int cols = chunks * 8;
    for (int col = tid; col < cols; col += kEwahToInt8Block) {
        uint32_t y[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const int j = t - (8 - Sa);
            y[t] = (j >= 0 && present[j]) ? planes32[static_cast<size_t>(j) * wpad * 2 + col] : 0u;
        }
        transpose8x8(y);
        uint4* dst = reinterpret_cast<uint4*>(out32 + (static_cast<size_t>(row) * cols + col) * 8);
        dst[0] = make_uint4(y[0], y[1], y[2], y[3]);
        dst[1] = make_uint4(y[4], y[5], y[6], y[7]);
    }
}

static unsigned stream_groups(int64_t R, int key_tiles) { return static_cast<unsigned>(((R + 15) / 16 + key_tiles - 1) / key_tiles); }
// one workgroup per CU at most: more waves each streaming their own chunks; else 8 and several workgroups
static int stream_waves(unsigned groups, int chunks, int slot) {
    int waves = groups <= 256 ? 16 : 8;
    if (waves > chunks) waves = chunks;          // one chunk per wave and pass at least
    if (waves < slot / 64) waves = slot / 64;    // the chain needs one lane per output
    return waves > 16 ? 16 : waves;
}
// Two key tiles per workgroup halve the query re-reads once there are enough tiles to fill the GPU.  With two tiles of queries besides,
// the sums take 4 KiB a chunk and the operands more than the registers a wave has.  us, one key tile and two: a dot of 16 x 8192 x
// 32768 49.3, 43.5, 16 x 4096 x 65536 49.5, 45.2; 32 x 4096 x 65536 65.0, 69.1, 32 x 4096 x 16384 15.6, 16.4, 32 x 8192 x 16384
// 33.7, 34.0, 32 x 12288 x 32768 94.4, 97.7, 17 x 16384 x 16384 57.3, 54.9; with the build inside 17 x 1024 x 16384 9.6, 14.8, 24 x 2048 x 16384 11.9, 16.9, 17 x 8192 x 16384 33.1, 38.4.
static int stream_key_tiles(int64_t Q, int64_t R) { return Q <= 16 && (R + 15) / 16 >= 1024 ? 2 : 1; }
void stream_launch_shape(int64_t Q, int64_t R, int chunks, unsigned* groups, int* waves) {
    const int kt = stream_key_tiles(Q, R);
    *groups = stream_groups(R, kt);
    *waves = stream_waves(*groups, chunks, kt * (Q <= 16 ? 1 : 2) * 256);
}

template <int NT, int KT>
static void launch_mfma_stream(const int8_t* A8, const float* qscale, int stride, const uint64_t* B, const float* Bw,
                               int chunks, int64_t R, int64_t Q, int down_shift, float scale_inv, int64_t R_total,
                               float* out, int32_t* chunk_ints, const float* bias, hipStream_t st) {
    constexpr int kSlot = KT * NT * 256;
    dim3 grid(stream_groups(R, KT), static_cast<unsigned>((Q + 16 * NT - 1) / (16 * NT)));
    const int waves = stream_waves(grid.x * grid.y, chunks, kSlot);
    constexpr int kChunkBytes = (kSlot + NT * 16) * 4;
    const size_t turn = kSlot < 512 && t_coop == nullptr ? static_cast<size_t>(waves) * 2048 : 0;
    int pass_chunks = kStreamLdsInts / kSlot;
    // 8 waves: two workgroups a CU
    if (turn != 0 && waves == 8 && pass_chunks * kChunkBytes + turn > 80 * 1024)
        pass_chunks = (80 * 1024 - static_cast<int>(turn)) / kChunkBytes / 8 * 8;
    if (pass_chunks > chunks) pass_chunks = chunks;
    const size_t lds = static_cast<size_t>(pass_chunks) * kChunkBytes + turn;
#define BSI_STREAM_GO(INTS, BUILD, COOP)                                                                                      \
    do {                                                                                                                      \
        static LdsOptIn once;                                                                                                 \
        if (lds > 64 * 1024) lds_opt_in(once, reinterpret_cast<const void*>(&dot_mfma_stream_kernel<NT, KT, INTS, BUILD>), kStreamLds); \
        launch((dot_mfma_stream_kernel<NT, KT, INTS, BUILD>), grid, dim3(waves * 64), lds, st, A8, qscale, stride,            \
               reinterpret_cast<const unsigned long long*>(B), Bw, chunks, pass_chunks, R, Q, down_shift, scale_inv, R_total, \
               out, chunk_ints, bias, t_out_dtype, COOP);                                                                     \
    } while (0)
    if (chunk_ints) BSI_STREAM_GO(true, 0, 0);
    else if (t_coop == nullptr) BSI_STREAM_GO(false, 0, 0);
    else {
        CoopBuild coop = *t_coop;
        grid.x = coop_groups(grid.x, R, coop, waves);
        coop.shares = coop_shares(grid.x, coop.by_row ? coop.rows : coop.rows * coop.chunks, coop.shares);
        if (coop.row_per_wave) BSI_STREAM_GO(false, 2, coop);
        else BSI_STREAM_GO(false, 1, coop);
    }
#undef BSI_STREAM_GO
}

void launch_mfma_stream_by_shape(const int8_t* A8, const float* qscale, int stride, const uint64_t* B, const float* Bw,
                                 int chunks, int64_t R, int64_t Q, int down_shift, float scale_inv, int64_t R_total,
                                 float* out, int32_t* chunk_ints, const float* bias, hipStream_t st) {
#define BSI_STREAM_ARGS A8, qscale, stride, B, Bw, chunks, R, Q, down_shift, scale_inv, R_total, out, chunk_ints, bias, st
    if (Q > 16) launch_mfma_stream<2, 1>(BSI_STREAM_ARGS);
    else if (stream_key_tiles(Q, R) == 2) launch_mfma_stream<1, 2>(BSI_STREAM_ARGS);
    else launch_mfma_stream<1, 1>(BSI_STREAM_ARGS);
#undef BSI_STREAM_ARGS
}

// Launch shape of the fused few-rows kernel: key tiles per workgroup, waves, and how many (chunk, row) items of the
// query build a wave takes up front (loads issued before the key loads; the rest go one at a time, each waiting for
// its own loads).
struct FusedPlan {
    int key_tiles, waves, upfront, per_wave;
    unsigned grid;
};
static FusedPlan fused_plan(int64_t Q, int chunks, int64_t R) {
    FusedPlan p;
    const int64_t ntiles = (R + 15) / 16;
    p.key_tiles = ntiles >= 1024 ? 2 : 1;  // two key tiles per workgroup once the GPU is full
    p.grid = static_cast<unsigned>((ntiles + p.key_tiles - 1) / p.key_tiles);
    p.waves = (p.grid <= 256) ? 16 : 8;  // as the few-rows kernel: one workgroup per CU gets more waves
    if (p.waves > chunks) p.waves = chunks;
    if (p.waves < p.key_tiles * 4) p.waves = p.key_tiles * 4;
    p.per_wave = static_cast<int>((static_cast<int64_t>(chunks) * Q + p.waves - 1) / p.waves);
    const int cap = p.key_tiles == 1 ? 4 : 2;
    p.upfront = p.per_wave <= 1 ? 1 : (p.per_wave <= 2 ? 2 : cap);
    return p;
}

template <typename T, int KT, int NI, bool kVec>
static void launch_stream_fused(const FusedPlan& plan, const T* x, int64_t d, double dec_scale, int slices, const uint64_t* B,
                                const float* Bw, int chunks, int64_t R, int Q, float scale_inv, int64_t R_total, float* out,
                                const float* bias, hipStream_t st) {
    constexpr int kSlot = KT * 256;
    // LDS: the query image and scales of all chunks, then as many chunk accumulators as fit beside them
    const size_t query_bytes = static_cast<size_t>(chunks) * Q * (256 + sizeof(float));
    int pass_chunks = kStreamLdsInts / kSlot;
    const int fit = static_cast<int>((150 * 1024 - query_bytes) / (kSlot * sizeof(int)));
    if (pass_chunks > fit) pass_chunks = fit;
    if (pass_chunks > chunks) pass_chunks = chunks;
    const size_t lds = static_cast<size_t>(pass_chunks) * kSlot * sizeof(int) + query_bytes;
    static LdsOptIn once0;
    lds_opt_in(once0, reinterpret_cast<const void*>(&dot_mfma_stream_fused_kernel<T, KT, NI, kVec>), 160 * 1024);
    const int narrow = integer_decimal_scale(dec_scale) != 0 ? 1 : 0;
    launch((dot_mfma_stream_fused_kernel<T, KT, NI, kVec>), dim3(plan.grid), dim3(plan.waves * 64), lds, st, x, d,
                       dec_scale, narrow, slices, reinterpret_cast<const unsigned long long*>(B), Bw, chunks, pass_chunks,
                       R, Q, scale_inv, R_total, out, bias, t_out_dtype);
}

template <typename T>
static void launch_stream_fused_t(const T* x, int64_t d, double dec_scale, int slices, const uint64_t* B, const float* Bw,
                                  int chunks, int64_t R, int Q, float scale_inv, int64_t R_total, float* out,
                                  const float* bias, hipStream_t st) {
    const FusedPlan p = fused_plan(Q, chunks, R);
    // a lane's four consecutive activations in one load where every row allows it
    const bool vec = d % 4 == 0 && reinterpret_cast<uintptr_t>(x) % (4 * sizeof(T)) == 0;
#define BSI_FUSED_GO(KT, NI)                                                                                              \
    {                                                                                                                     \
        if (vec) launch_stream_fused<T, KT, NI, true>(p, x, d, dec_scale, slices, B, Bw, chunks, R, Q, scale_inv, R_total, out, bias, st); \
        else launch_stream_fused<T, KT, NI, false>(p, x, d, dec_scale, slices, B, Bw, chunks, R, Q, scale_inv, R_total, out, bias, st);    \
    }
    if (p.key_tiles == 2) {
        if (p.upfront == 1) BSI_FUSED_GO(2, 1)
        else BSI_FUSED_GO(2, 2)
    } else {
        if (p.upfront == 1) BSI_FUSED_GO(1, 1)
        else if (p.upfront == 2) BSI_FUSED_GO(1, 2)
        else BSI_FUSED_GO(1, 4)
    }
#undef BSI_FUSED_GO
}

}  // namespace bsi

using namespace bsi;

extern "C" int bsi_hip_linear_few_rows_upfront(int64_t Q, int64_t d, int64_t R) {
    if (Q < 1 || Q > kFusedMaxQ || d < 1 || R < 1) return 0;
    const FusedPlan p = fused_plan(Q, static_cast<int>((d + 255) / 256), R);
    return p.per_wave <= p.upfront ? 1 : 0;
}

// A build that every workgroup repeats costs a round of loads for each item a wave has beyond those up front; the one that an XCD's
// workgroups share costs a wait.  us, each (rows x width x keys): 4 x 8192 x 8192 20.0, 11.9; 4 x 5120 x 5120 13.5, 8.7; 4 x 4096 x 11008 14.5,
// 11.7; 3 x 4096 x 5120 9.6, 8.1; 3 x 4096 x 11008 12.2, 11.7; 2 x 8192 x 8192 14.6, 11.9; 2 x 5120 x 5120 9.5, 8.7; with two key tiles a
// workgroup 2 x 4096 x 16384 12.9, 11.8; 3 x 2304 x 16384 9.9, 8.9 -- where the loads hide it, or one more: 4 x 4096 x 4096 6.8, 7.4; 2 x
// 4096 x 11008 10.2, 11.5; 1 x 8192 x 8192 11.2, 11.8; 2 x 2304 x 16384 8.5, 8.8.
extern "C" int bsi_hip_linear_few_rows_shares(int64_t Q, int64_t d, int64_t R) {
    if (Q < 1 || Q > kFusedMaxQ || d < 1 || R < 1) return 0;
    const FusedPlan p = fused_plan(Q, static_cast<int>((d + 255) / 256), R);
    return p.per_wave > p.upfront + (p.key_tiles == 2 ? 1 : 0) ? 1 : 0;
}

static int linear_few_rows(const void* x, int dtype, int64_t Q, int64_t d, int decimal_places, int fixed_bits,
                           const uint64_t* B_tiled, const float* Bw, int Sb, int64_t R, float scale_inv, int64_t R_total,
                           const float* bias, float* out, void* stream) {
    BSI_REQUIRE(Q >= 0 && R >= 0 && d >= 1, "bad shape");
    BSI_REQUIRE(Q <= kFusedMaxQ, "the fused few-rows kernel takes at most %d query rows (got %lld)", kFusedMaxQ,
                static_cast<long long>(Q));
    BSI_REQUIRE(fixed_bits >= 2 && fixed_bits <= 8, "fixed_bits must be in [2, 8] (got %d)", fixed_bits);
    BSI_REQUIRE(R_total >= R, "R_total must be >= R");
    if (Sb != 6) return fail(BSI_ERR_UNSUPPORTED, "the fused few-rows kernel reads 6-plane tiled keys (got Sb = %d)", Sb);
    const int W64 = static_cast<int>((d + 63) / 64);
    if (W64 % 4 != 0)
        return fail(BSI_ERR_UNSUPPORTED, "chunk scales need a multiple of 4 words per slice (d = %lld)", static_cast<long long>(d));
    if (Q == 0 || R == 0) return BSI_OK;
    BSI_REQUIRE(x && B_tiled && Bw && out, "null pointer");
    const int chunks = W64 / 4;
    if (static_cast<size_t>(chunks) * Q * (256 + sizeof(float)) > kFusedQueryLdsBytes)
        return fail(BSI_ERR_UNSUPPORTED, "%lld rows of %lld elements do not fit the kernel's LDS query buffer (%zu bytes)",
                    static_cast<long long>(Q), static_cast<long long>(d), kFusedQueryLdsBytes);
    const double dec_scale = pow(10.0, static_cast<double>(decimal_places));
    hipStream_t st = as_stream(stream);
#define BSI_FUSED(T)                                                                                                \
    launch_stream_fused_t<T>(static_cast<const T*>(x), d, dec_scale, fixed_bits, B_tiled, Bw, chunks, R, static_cast<int>(Q), \
                             scale_inv, R_total, out, bias, st);
    if (dtype == BSI_DTYPE_F32) { BSI_FUSED(float) }
    else if (dtype == BSI_DTYPE_F16) { BSI_FUSED(__half) }
    else if (dtype == BSI_DTYPE_BF16) { BSI_FUSED(__hip_bfloat16) }
    else return fail(BSI_ERR_INVALID, "unknown dtype %d", dtype);
#undef BSI_FUSED
    BSI_LAUNCH_CHECK("dot_mfma_stream_fused_kernel");
    return BSI_OK;
}

extern "C" int bsi_hip_linear_few_rows(const void* x, int dtype, int64_t Q, int64_t d, int decimal_places, int fixed_bits,
                                       const uint64_t* B_tiled, const float* Bw, int Sb, int64_t R, float scale_inv,
                                       int64_t R_total, const float* bias, float* out, void* stream) {
    return linear_few_rows(x, dtype, Q, d, decimal_places, fixed_bits, B_tiled, Bw, Sb, R, scale_inv, R_total, bias, out, stream);
}

extern "C" int bsi_hip_linear_few_rows_out(const void* x, int dtype, int64_t Q, int64_t d, int decimal_places, int fixed_bits,
                                           const uint64_t* B_tiled, const float* Bw, int Sb, int64_t R, float scale_inv,
                                           int64_t R_total, const float* bias, void* out, int out_dtype, void* stream) {
    BSI_REQUIRE(out_dtype == BSI_DTYPE_F32 || out_dtype == BSI_DTYPE_F16 || out_dtype == BSI_DTYPE_BF16, "unknown dtype code %d", out_dtype);
    t_out_dtype = out_dtype;
    const int rc = linear_few_rows(x, dtype, Q, d, decimal_places, fixed_bits, B_tiled, Bw, Sb, R, scale_inv, R_total, bias,
                                   static_cast<float*>(out), stream);
    t_out_dtype = BSI_DTYPE_F32;
    return rc;
}

// Launch of the inline-decode kernel for Q queries (groups of 16 along grid.y), or BSI_ERR_UNSUPPORTED when the
// planes of a group do not fit LDS.
static int launch_stream_ewah(const uint64_t* comp_words, const int64_t* comp_off, const int32_t* comp_len, int Sa, int W64,
                              const float* A_chunk_scales, int A_scale_stride, const uint64_t* B_tiled, const float* Bw,
                              int64_t R, int64_t Q, float scale_inv, int64_t R_total, const float* bias, float* out,
                              int32_t* chunk_ints, hipStream_t st) {
    const int chunks = (W64 + 3) / 4;
    const int group = static_cast<int>(Q < kEwahQueriesPerGroup ? Q : kEwahQueriesPerGroup);
    const size_t plane_bytes = ewah_plane_region(group, Sa, chunks * 4) + 128;
    if (plane_bytes > 120 * 1024)
        return fail(BSI_ERR_UNSUPPORTED, "%d words per slice do not fit the LDS plane buffer of the inline-decode kernel", W64);
    int pass_chunks = static_cast<int>((kStreamLdsInts * sizeof(int) < 156 * 1024 - plane_bytes
                                            ? kStreamLdsInts * sizeof(int)
                                            : 156 * 1024 - plane_bytes) / 1024);
    if (pass_chunks > chunks) pass_chunks = chunks;
    const size_t lds = plane_bytes + static_cast<size_t>(pass_chunks) * 1024;
    int waves = chunks < 16 ? chunks : 16;
    if (waves < 4) waves = 4;
    const dim3 grid(static_cast<unsigned>((R + 15) / 16), static_cast<unsigned>((Q + kEwahQueriesPerGroup - 1) / kEwahQueriesPerGroup));
    static LdsOptIn once0;
    lds_opt_in(once0, reinterpret_cast<const void*>(&dot_mfma_stream_ewah_kernel<true>), 160 * 1024);
    static LdsOptIn once1;
    lds_opt_in(once1, reinterpret_cast<const void*>(&dot_mfma_stream_ewah_kernel<false>), 160 * 1024);
    const int down_shift = 16 - Sa - 6;
#define BSI_EWAH_ARGS reinterpret_cast<const unsigned long long*>(comp_words), reinterpret_cast<const long long*>(comp_off), \
                      comp_len, Sa, W64, A_chunk_scales, A_scale_stride, reinterpret_cast<const unsigned long long*>(B_tiled), \
                      Bw, chunks, pass_chunks, R, Q, group, down_shift, scale_inv, R_total, bias, out, chunk_ints
    if (chunk_ints) launch((dot_mfma_stream_ewah_kernel<true>), grid, dim3(waves * 64), lds, st, BSI_EWAH_ARGS);
    else launch((dot_mfma_stream_ewah_kernel<false>), grid, dim3(waves * 64), lds, st, BSI_EWAH_ARGS);
#undef BSI_EWAH_ARGS
    BSI_LAUNCH_CHECK("dot_mfma_stream_ewah_kernel");
    return BSI_OK;
}

extern "C" int bsi_hip_dot_ewah_query(const uint64_t* comp_words, const int64_t* comp_off, const int32_t* comp_len,
                                      int Sa, int W64, const float* A_chunk_scales, int A_scale_stride,
                                      const uint64_t* B_tiled, const float* Bw, int Sb, int64_t R, float scale_inv,
                                      float* out, int32_t* chunk_ints, void* stream) {
    BSI_REQUIRE(R >= 0 && W64 >= 1, "bad shape");
    BSI_REQUIRE(Sa >= 2 && Sa <= 8, "Sa must be in [2, 8] (got %d)", Sa);
    if (Sb != 6) return fail(BSI_ERR_UNSUPPORTED, "the inline-decode kernel reads 6-plane tiled keys (got Sb = %d)", Sb);
    if (R == 0) return BSI_OK;
    BSI_REQUIRE(comp_words && comp_off && comp_len && A_chunk_scales && B_tiled && Bw && out, "null pointer");
    const int chunks = (W64 + 3) / 4;
    BSI_REQUIRE(A_scale_stride == chunks || A_scale_stride == 1,
                "chunk scale stride mismatch: got %d expected %d (or 1 for a row scale)", A_scale_stride, chunks);
    return launch_stream_ewah(comp_words, comp_off, comp_len, Sa, W64, A_chunk_scales, A_scale_stride, B_tiled, Bw, R, 1,
                              scale_inv, R, nullptr, out, chunk_ints, as_stream(stream));
}

extern "C" size_t bsi_hip_dot_ewah_batch_workspace_bytes(int64_t Q, int W64) {
    return bsi_hip_dot_workspace_bytes(Q, W64, BSI_CORE_MFMA);
}

extern "C" int bsi_hip_dot_ewah_batch(const uint64_t* comp_words, const int64_t* comp_off, const int32_t* comp_len, int Sa,
                                      int W64, const float* A_chunk_scales, int A_scale_stride, const uint64_t* B,
                                      int b_layout, const float* Bw, int Sb, int64_t R, int64_t Q, float scale_inv,
                                      int64_t R_total, const float* bias, float* out, int32_t* chunk_ints, void* workspace,
                                      size_t workspace_bytes, void* stream) {
    BSI_REQUIRE(Q >= 0 && R >= 0 && W64 >= 1 && R_total >= R, "bad shape");
    BSI_REQUIRE(Sa >= 2 && Sa <= 8 && Sb >= 2 && Sb <= 8, "the matrix-core dot needs Sa, Sb in [2, 8] (got %d, %d)", Sa, Sb);
    if (Q == 0 || R == 0) return BSI_OK;
    BSI_REQUIRE(comp_words && comp_off && comp_len && A_chunk_scales && B && Bw && out, "null pointer");
    const int chunks = (W64 + 3) / 4;
    BSI_REQUIRE(A_scale_stride == chunks || A_scale_stride == 1,
                "chunk scale stride mismatch: got %d expected %d (or 1 for row scales)", A_scale_stride, chunks);
    hipStream_t st = as_stream(stream);
    // A few rows against the packed planes: each workgroup can afford to expand the queries itself -- the decode is part of the
    // dot kernel's load stage.  Every workgroup repeats it, though, and more than 16 rows stream the keys twice, so with more than
    // eight rows, or eight's worth of 4096 elements, a launch for the decode pays for itself.  us a pass of build and dot, decode
    // inside and in a launch ahead (rows x width x keys): 4 x 4096 x 4096 27.2, 29.0; 8 x 2048 x 2048 27.8, 29.1; 8 x 4096 x 4096
    // 28.9, 28.9 -- beyond: 4 x 8192 x 1024 31.2, 29.6; 8 x 8192 x 1024 32.8, 30.2; 12 x 768 x 768 33.7, 29.5; 12 x 2048 x 2048
    // 30.8, 29.1; 16 x 2048 x 8192 33.4, 28.9; 32 x 1600 x 4800 42.2, 30.9; 32 x 4096 x 4096 39.5, 31.1.  Calls without a workspace
    // have no choice.
    const int64_t group = Q < kEwahQueriesPerGroup ? Q : kEwahQueriesPerGroup;
    const size_t need = bsi_hip_dot_ewah_batch_workspace_bytes(Q, W64);
    const bool decode_ahead = (Q > 8 || Q * chunks >= 128) && workspace != nullptr && workspace_bytes >= need &&
                              (reinterpret_cast<uintptr_t>(workspace) & 15) == 0;
    if (!decode_ahead && Q <= kStreamMaxQ && b_layout == BSI_LAYOUT_TILED16 && Sb == 6 &&
        ewah_plane_region(static_cast<int>(group), Sa, chunks * 4) + 128 <= 120 * 1024)
        return launch_stream_ewah(comp_words, comp_off, comp_len, Sa, W64, A_chunk_scales, A_scale_stride, B, Bw, R, Q,
                                  scale_inv, R_total, bias, out, chunk_ints, st);
    // Many rows: every key-tile workgroup of the compute-bound kernel reads the whole query tile, so expanding the
    // streams there would repeat the decode and the plane -> int8 recombination once per key tile (32 times at
    // Q512 x R2048).  The call's load stage therefore runs once, as a launch of its own: streams -> int8 query
    // image in the workspace (the verbatim planes are never materialised), then the dot on that image.
    BSI_REQUIRE(workspace != nullptr && workspace_bytes >= need, "%zu bytes of workspace needed for the int8 query image (got %zu)",
                need, workspace_bytes);
    BSI_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 15) == 0, "workspace must be 16-byte aligned");
    const size_t lds = static_cast<size_t>(Sa) * chunks * 4 * 8 + 64;
    if (lds > 150 * 1024)
        return fail(BSI_ERR_UNSUPPORTED, "%d words per slice do not fit the LDS plane buffer of the stream decoder", W64);
    static LdsOptIn once;
    lds_opt_in(once, reinterpret_cast<const void*>(&ewah_streams_to_int8_kernel), 160 * 1024);
    launch(ewah_streams_to_int8_kernel, dim3(static_cast<unsigned>(Q)), dim3(kEwahToInt8Block), lds, st,
                       reinterpret_cast<const unsigned long long*>(comp_words), reinterpret_cast<const long long*>(comp_off),
                       comp_len, Sa, W64, chunks, static_cast<uint32_t*>(workspace));
    BSI_LAUNCH_CHECK("ewah_streams_to_int8_kernel");
    return dot_with_bias(nullptr, static_cast<const int8_t*>(workspace), A_chunk_scales, A_scale_stride, Sa, W64, B, b_layout,
                         Bw, Sb, R, Q, scale_inv, R_total, out, chunk_ints, BSI_CORE_MFMA, nullptr, 0, stream, bias);
}
