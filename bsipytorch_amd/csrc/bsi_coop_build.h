// The query build of a small linear layer inside its dot's launch.
//
// A layer of a few rows is two launches, the query build and the dot, and the build is nothing but a launch: 2.2 us on the GPU
// and 2.7 on the host for a fraction of a microsecond of work.  Building per workgroup repeats the work for every key tile;
// building once for the device needs what one XCD wrote to become visible to the others.  So every XCD builds a copy of its
// own: the workgroups on it take a share each, all of them read the copy through the L2 they share, and a share is announced
// by a flag behind it.
//
// No workgroup depends on another one being resident.  A share's bytes do not depend on who builds it, so a workgroup that
// has waited kCoopPatience for a share builds it itself: beside kernels that hold the CUs, most shares of a copy may belong to workgroups
// that have not begun.  Every CU of an XCD begins at another missing share, and between two a workgroup looks at all flags.  us a layer of
// 16 x 4096 x 4096 beside one of 4096 x 4096 x 16384 on another stream (256 workgroups with all LDS of a CU each), median of 36: 150 with
// a patience of 20 us and the lowest share first for all, 106 from different shares, 83 with 10 us, 64 to 71 with 5, 62 with 3; layers of a
// few tiles 35 to 50 in all forms.  On an idle GPU a build takes 2 to 5 us from the first workgroup's begin, and a share is waited for from
// the end of the own one.  (Half the patience for every further share: 78, but the few-rows kernel then keeps other arguments in
// registers: 12 x 4096 x 11008 12.1, 11.5; 16 x 5376 x 7168 10.2, 10.4; 12 x 2048 x 8192 6.3, 6.5.)  Flags hold the launch's number, which no other launch has: nothing
// is cleared between launches, and flags of earlier ones mean nothing.
//
// What a reader relies on, since neither side of a flag is more than a relaxed access (an agent-scope release writes the L2
// back: the flags come 1 to 2 us later; an agent-scope acquire also drops L2 lines: 16 x 4096 x 4096 7.4 -> 8.8 us, 15 x 2560
// x 5888 7.3 -> 9.5):
//  - A store is complete (vmcnt) when the XCD's L2 has it, and a copy is written and read by workgroups of its own XCD only:
//    the index is XCC_ID, in the build and in the reads.
//  - No L1 holds a line of a copy that another CU has written in this launch.  L1s and scalar caches are invalidated when a
//    kernel starts, as every kernel that reads what an earlier one wrote needs; and within the launch nothing loads from a copy
//    before all its flags are there, so that the first load of a line fetches it from the L2.  That is why coop_build hands
//    out the copy's address only when it returns, and why ahead() must not load from `area`: a load there would compile and
//    read right most of the time.
//  - Flags are read past the L1 (agent scope) and share no line with a copy; a copy's lines belong to it alone.
//  - Lines of a copy that several CUs write lose no byte of it: an L1 writes through the bytes that were stored and no others, the
//    L2 puts them together, and an L1 answers with no byte of a line that it has not fetched or written itself.  Such are the lines of
//    the scales, four bytes a wave, and, in the order of the few-rows kernel's operands (kFragments), those of the image: a line of
//    128 bytes holds 16 of each of eight rows, written by up to eight waves of as many CUs.  In rows one after the other an item's 256
//    bytes are two lines, and one wave's.
// Inside a launch of 16 rows of 4096 the workgroups have the whole build 3.2 us after the first wave has begun (wall clock stamps:
// 1.3 until a wave has its chunk and has quantised it, 0.9 to the flag, the stamps' own stores among that, 0.6 to the last
// share); 2.3 us at 16 rows of 512.  That is as long as the launch it replaces, but for the host.
#pragma once
#include "bsi_quant_device.h"

namespace bsi {

constexpr int kXcds = 8;
constexpr int kCoopShares = 32;       // shares of a copy at most: one workgroup for each CU of an XCD
constexpr int kCoopHeld = 8;          // chunks of a row that a wave builds by itself
constexpr int kCoopMaxItems = 1024;   // (row, chunk) items: 256 bytes of image and a scale each
constexpr size_t kCoopFlagBytes = kXcds * kCoopShares * sizeof(unsigned long long);
constexpr size_t kCoopCopyBytes = static_cast<size_t>(kCoopMaxItems) * (BSI_CHUNK_ELEMS + sizeof(float));
constexpr size_t kCoopBytes = kCoopFlagBytes + kXcds * kCoopCopyBytes;
static_assert(kCoopFlagBytes % 128 == 0 && kCoopCopyBytes % 128 == 0, "flags and copies share no cache line");
constexpr int kCoopPatience = 500;  // ticks of the 100 MHz clock: 5 us

struct CoopBuild {
    const void* x;
    unsigned char* area;        // kCoopBytes: flags, then the copies (image, scales)
    unsigned long long launch;  // this launch's number
    long long d;
    double dec_scale;
    float scale;
    int dtype, vec;             // BSI_DTYPE_*; rows can be loaded a quad at a time
    int rows, chunks, slices;
    int by_row;                 // one scale a row instead of one a chunk
    int row_per_wave;           // by_row: a wave builds a row (of kCoopHeld chunks at most) by itself: instances of their own
    int shares;                 // of a copy: chunk scales split the items, row scales the rows (ahead of the launch: asked for, or 0)
    int patience;               // ticks until a workgroup builds what it waits for
};

// Workgroups of a launch whose dot has `groups`: a few tiles leave most CUs idle, and their few workgroups would build round after
// round, so there are as many as a build of one round has shares of waves (row scales: of rows), one for each CU at most.  The
// kernels tell those without a tile by themselves.  33 x 768 x 768 is 12 tiles and 99 items: 9.7 us in two launches, 6.4 in one.
// Not for fewer than kCoopMinKeys keys: those are fed what wider layers beside them are fed, and take over its build, which a build
// inside the launch is not (18 x 512 x 64 behind a layer of the same tensor: one launch either way).
constexpr int kCoopMinKeys = 256;
inline unsigned coop_groups(unsigned groups, int64_t keys, const CoopBuild& b, int waves) {
    if (keys < kCoopMinKeys) return groups;
    const int pieces = b.by_row ? b.rows : b.rows * b.chunks, a_share = b.by_row && !b.row_per_wave ? 1 : waves;
    const int shares = (pieces + a_share - 1) / a_share < kCoopShares ? (pieces + a_share - 1) / a_share : kCoopShares;
    return groups < static_cast<unsigned>(shares * kXcds) ? static_cast<unsigned>(shares * kXcds) : groups;
}
// Shares of a copy for a grid of `groups` workgroups, which go to the XCDs in turn; or as many as are asked for (a test's shares
// that no workgroup owns).
inline int coop_shares(unsigned groups, int pieces, int asked = 0) {
    int shares = asked > 0 ? asked : static_cast<int>(groups / kXcds);
    if (shares > kCoopShares) shares = kCoopShares;
    if (shares > pieces) shares = pieces;
    return shares < 1 ? 1 : shares;
}

// Where dword `lane` of a (row, chunk) item lies in a copy, in dwords.  kFragments: in the order in which the few-rows kernel
// takes its operands -- 16 rows at a time, then chunk, MFMA, quarter of its 64 elements, row -- so that each of its loads is one
// run of up to 1 KiB; from rows one after the other a load takes 16 bytes out of every 64 of 16 rows, 32 lines.
template <bool kFragments>
__device__ __forceinline__ int coop_image_at(const CoopBuild& b, int row, int chunk, int lane) {
    if (!kFragments) return (row * b.chunks + chunk) * 64 + lane;
    const int first = row & ~15, rows = b.rows - first < 16 ? b.rows - first : 16;
    return first * b.chunks * 64 + (((chunk * 4 + (lane >> 2 & 3)) * 4 + (lane >> 4)) * rows + (row & 15)) * 4 + (lane & 3);
}

// Where its scale lies: beside those of the chunk's other rows (kFragments), or of the row's other chunks.
template <bool kFragments>
__device__ __forceinline__ int coop_scale_at(const CoopBuild& b, int row, int chunk) {
    if (!kFragments) return row * b.chunks + chunk;
    const int first = row & ~15, rows = b.rows - first < 16 ? b.rows - first : 16;
    return first * b.chunks + chunk * rows + (row & 15);
}

// Row scales: the row's largest magnitude over the waves, then its quantised chunks, a row of the share after the other.
// kRowPerWave: a wave has a row of up to kCoopHeld chunks to itself, all its loads at once and no barrier, so that a share takes
// as long as one row for as many rows as the workgroup has waves.  An instance of its own: with it beside the other form the
// dot's kernels take 105 registers for 68 (121 x 512 x 14848 8.4 -> 8.9 us, 12 x 1600 x 4800 6.5 -> 6.9).
template <typename T, bool kVec, bool kFragments, bool kRowPerWave>
__device__ void coop_build_share(const CoopBuild& b, int share, int wave, int nwaves, int lane, uint32_t* __restrict__ image,
                                 float* __restrict__ scales, unsigned* __restrict__ wave_max) {
    const ChunkLane cl = chunk_lane(lane);
    const QuantRange range = quant_range(b.slices);
    const T* const x = static_cast<const T*>(b.x);
    if (!kRowPerWave && !b.by_row) {
        const int items = b.rows * b.chunks;
        const int first = items * share / b.shares, last = items * (share + 1) / b.shares;
        auto load = [&](int item, float (&v)[4]) {
            const int row = item / b.chunks;
            load_chunk_quad<T, kVec>(x + row * b.d, b.d, item - row * b.chunks, cl, v);
        };
        auto emit = [&](int item, const float (&v)[4]) {
            const int row = item / b.chunks;
            const unsigned mx = wave_max_u32(quad_max_bits(v));
            int shift;
            uint32_t bytes;
            if (mx < kQuantWideBits) {
                shift = quant_shift(mx, b.scale, b.slices);
                bytes = quantise_quad<T>(v, b.scale, shift, range);
            } else {
                shift = compute_shift(wave_max_u64(quad_max_wide(v, b.dec_scale)), 0.0, 1, b.slices, 0.0f);
                bytes = quantise_quad_wide(v, b.dec_scale, shift, b.slices);
            }
            image[coop_image_at<kFragments>(b, row, item - row * b.chunks, lane)] = chunk_image_dword(bytes, cl);
            if (lane == 0) scales[coop_scale_at<kFragments>(b, row, item - row * b.chunks)] = static_cast<float>(1ULL << shift);
        };
#pragma unroll 1
        for (int item = first + wave; item < last; item += nwaves) {
            float v[4];
            load(item, v);
            emit(item, v);
        }
        return;
    }
    const int first = b.rows * share / b.shares, last = b.rows * (share + 1) / b.shares;
    if constexpr (kRowPerWave) {
#pragma unroll 1
        for (int row = first + wave; row < last; row += nwaves) {
            const T* const xrow = x + row * b.d;
            unsigned mx = kQuantWideBits;
            if constexpr (kVec) {
                float held[kCoopHeld][4];
#pragma unroll
                for (int c = 0; c < kCoopHeld; ++c) load_chunk_quad<T, true>(xrow, b.d, c, cl, held[c]);  // past the row: zeros
                mx = 0u;
#pragma unroll
                for (int c = 0; c < kCoopHeld; ++c) {
                    const unsigned m = quad_max_bits(held[c]);
                    mx = m > mx ? m : mx;
                }
                mx = wave_max_u32(mx);
                if (mx < kQuantWideBits) {
                    const int shift = quant_shift(mx, b.scale, b.slices);
                    if (lane == 0) scales[row] = static_cast<float>(1ULL << shift);
#pragma unroll
                    for (int c = 0; c < kCoopHeld; ++c)
                        if (c < b.chunks)
                            image[coop_image_at<kFragments>(b, row, c, lane)] = chunk_image_dword(quantise_quad<T>(held[c], b.scale, shift, range), cl);
                }
            }
            if (mx >= kQuantWideBits) {  // rare, as are rows that no quad can be loaded from: the general routine, a chunk at a time
                unsigned long long m64 = 0ULL;
#pragma unroll 1
                for (int c = 0; c < b.chunks; ++c) {
                    float v[4];
                    load_chunk_quad<T, kVec>(xrow, b.d, c, cl, v);
                    const unsigned long long m = quad_max_wide(v, b.dec_scale);
                    m64 = m > m64 ? m : m64;
                }
                const int shift = compute_shift(wave_max_u64(m64), 0.0, 1, b.slices, 0.0f);
                if (lane == 0) scales[row] = static_cast<float>(1ULL << shift);
#pragma unroll 1
                for (int c = 0; c < b.chunks; ++c) {
                    float v[4];
                    load_chunk_quad<T, kVec>(xrow, b.d, c, cl, v);
                    image[coop_image_at<kFragments>(b, row, c, lane)] = chunk_image_dword(quantise_quad_wide(v, b.dec_scale, shift, b.slices), cl);
                }
            }
        }
        return;
    }
#pragma unroll 1
    for (int row = first; row < last; ++row) {
        const T* const xrow = x + row * b.d;
        float held[4];
        load_chunk_quad<T, kVec>(xrow, b.d, wave, cl, held);  // past the row: zeros
        unsigned mx = quad_max_bits(held);
        for (int c = wave + nwaves; c < b.chunks; c += nwaves) {
            float v[4];
            load_chunk_quad<T, kVec>(xrow, b.d, c, cl, v);
            const unsigned m = quad_max_bits(v);
            mx = m > mx ? m : mx;
        }
        mx = wave_max_u32(mx);
        if (lane == 0) wave_max[wave] = mx;
        lds_barrier();
        for (int w = 0; w < nwaves; ++w) mx = wave_max[w] > mx ? wave_max[w] : mx;
        lds_barrier();
        const bool wide = mx >= kQuantWideBits;
        int shift = quant_shift(mx, b.scale, b.slices);
        if (wide) {  // rare: every wave looks at the whole row
            unsigned long long m64 = 0ULL;
            for (int c = 0; c < b.chunks; ++c) {
                float v[4];
                load_chunk_quad<T, kVec>(xrow, b.d, c, cl, v);
                const unsigned long long m = quad_max_wide(v, b.dec_scale);
                m64 = m > m64 ? m : m64;
            }
            shift = compute_shift(wave_max_u64(m64), 0.0, 1, b.slices, 0.0f);
        }
        if (wave == 0 && lane == 0) scales[row] = static_cast<float>(1ULL << shift);
        for (int c = wave; c < b.chunks; c += nwaves) {
            float v[4];
            if (c == wave) {
#pragma unroll
                for (int k = 0; k < 4; ++k) v[k] = held[k];
            } else {
                load_chunk_quad<T, kVec>(xrow, b.d, c, cl, v);
            }
            const uint32_t bytes = wide ? quantise_quad_wide(v, b.dec_scale, shift, b.slices) : quantise_quad<T>(v, b.scale, shift, range);
            image[coop_image_at<kFragments>(b, row, c, lane)] = chunk_image_dword(bytes, cl);
        }
    }
}

// Called by all waves of the workgroup (number `id` of the grid); 32 words of LDS at `shared`.  On return A8 and qscale point
// to the whole build, in the copy of the XCD the workgroup runs on.  ahead(): loads for after the build, of anything but the
// area, inside for any id.  Every wave but wave 0 issues them when the workgroup's share is built (a CU's loads return in order: not before),
// wave 0, which asks for the flags, when all shares are.
template <bool kFragments, bool kRowPerWave, typename F>
__device__ __forceinline__ void coop_build(const CoopBuild& b, unsigned id, unsigned* __restrict__ shared, const int8_t*& A8,
                                           const float*& qscale, F&& ahead) {
    const int lane = threadIdx.x & (BSI_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int nwaves = static_cast<int>(blockDim.x >> 6);
    const unsigned xcd = __builtin_amdgcn_s_getreg((3 << 11) | 20) & (kXcds - 1);  // XCC_ID, bits 0 .. 3
    unsigned long long* const flags = reinterpret_cast<unsigned long long*>(b.area) + xcd * kCoopShares;
    unsigned char* const copy = b.area + kCoopFlagBytes + xcd * kCoopCopyBytes;
    uint32_t* const image = reinterpret_cast<uint32_t*>(copy);
    float* const scales = reinterpret_cast<float*>(copy + static_cast<size_t>(kCoopMaxItems) * BSI_CHUNK_ELEMS);
    bool issued = false;
    auto build = [&](int share) {
        if (b.dtype == BSI_DTYPE_F32) {
            if (b.vec) coop_build_share<float, true, kFragments, kRowPerWave>(b, share, wave, nwaves, lane, image, scales, shared);
            else coop_build_share<float, false, kFragments, kRowPerWave>(b, share, wave, nwaves, lane, image, scales, shared);
        } else if (b.dtype == BSI_DTYPE_F16) {
            if (b.vec) coop_build_share<__half, true, kFragments, kRowPerWave>(b, share, wave, nwaves, lane, image, scales, shared);
            else coop_build_share<__half, false, kFragments, kRowPerWave>(b, share, wave, nwaves, lane, image, scales, shared);
        } else {
            if (b.vec) coop_build_share<__hip_bfloat16, true, kFragments, kRowPerWave>(b, share, wave, nwaves, lane, image, scales, shared);
            else coop_build_share<__hip_bfloat16, false, kFragments, kRowPerWave>(b, share, wave, nwaves, lane, image, scales, shared);
        }
        const int items = b.rows * b.chunks, had = items * (share + 1) / b.shares - items * share / b.shares;
        if (b.by_row || wave < had) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the wave's stores have reached the L2
        lds_barrier();
        if (wave != 0 && !issued) {
            ahead();
            issued = true;
        }
        // A plain store, as the share's are: it stops in the L2 that the workgroups of this XCD share, where their agent-scope
        // loads find it.  (An agent-scope store goes on to memory: the flags then come 1 to 2 us later.)
        if (threadIdx.x == 0) __hip_atomic_store(flags + share, b.launch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    int share = id / kXcds < static_cast<unsigned>(b.shares) ? static_cast<int>(id / kXcds) : -1;
    if (share < 0 && wave != 0) {
        ahead();
        issued = true;
    }
#pragma unroll 1
    for (;;) {
        if (share >= 0) build(share);
        if (wave == 0) {
            const unsigned long long since = wall_clock64();
            unsigned long long missing;
            for (;;) {
                const bool here = lane >= b.shares ||
                                  __hip_atomic_load(flags + (lane < kCoopShares ? lane : 0), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == b.launch;
                missing = __ballot(!here);
                if (missing == 0ULL || wall_clock64() - since > static_cast<unsigned>(b.patience)) break;
            }
            if (lane == 0) shared[0] = static_cast<unsigned>(missing);
        }
        lds_barrier();
        const unsigned missing = static_cast<unsigned>(__builtin_amdgcn_readfirstlane(static_cast<int>(shared[0])));
        lds_barrier();
        if (missing == 0u) break;
        // HW_ID, CU and shader engine: every CU of an XCD begins elsewhere, and neighbours (the first to be given work) far apart
        const unsigned cu = __builtin_amdgcn_s_getreg((7 << 11) | (8 << 6) | 4), from = ((cu & 7u) * 4u + (cu >> 5 & 3u)) * 13u % kCoopShares;
        share = static_cast<int>((__builtin_ctz(__builtin_rotateright32(missing, from)) + from) % kCoopShares);
    }
    if (!issued) ahead();
    asm volatile("" ::: "memory");
    A8 = reinterpret_cast<const int8_t*>(copy);
    qscale = scales;
}

}  // namespace bsi
