// The matrix-core dot on the cached int8 image of the keys (the compute-bound calls), its probe of the L2 -> LDS
// path, the timeline stamps, and the decimal-mode dot on int8 digit images that runs on the same kernel.
// Shapes in the comments are rows x width x keys.
#include "bsi_coop_build.h"
#include "bsi_dot_internal.h"

#include <type_traits>

namespace bsi {

// process-wide options set through bsi_hip_set_option (meanings beside their declarations in bsi_dot_internal.h)
std::atomic<int> g_i8_tile{0};
std::atomic<int> g_digits_route{0};

// ------------------------------------------------------------------ MFMA core on the cached int8 key image
//
// Compute-bound shapes (hundreds of query rows) pay for the plane -> int8 recombination of the keys
// on the vector ALU in every workgroup that touches a key tile.  A keyset can therefore carry,
// next to its packed planes, the recombined int8 image of the same integers (built once by
// bsi_hip_planes_to_int8, 1 byte per weight); this kernel contracts that image with the int8
// query image.
//   * workgroup = 128 keys x 128 queries over all chunks; 8 MFMA waves of 64 keys x 32 queries
//     and 4 loader waves (one per SIMD).  Only the loader waves issue global loads: a wave that
//     issues them blocks while the memory queue is full, which the MFMA waves must never do;
//   * LDS is a ring of four half-chunk stages (keys 128 x 128 B + queries 128 x 128 B = 32 KiB
//     each), filled by buffer loads that write LDS directly (a loader wave issues 4 + 4 per
//     stage, 1 KiB each); the 16-byte columns of a row are XOR-swizzled with (row >> 1) & 7 so
//     that the 16 rows a ds_read_b128 touches hit distinct banks;
//   * loads of half h+3 are issued when half h starts; the wait before the barrier that ends half
//     h only covers the loads of half h+1, so two stages stay in flight across barriers;
//   * the fp32 epilogue of chunk c-1 (one cvt + one fma per output and chunk, in chunk order)
//     is interleaved element by element with the MFMAs of chunk c (two accumulator sets).

// Peak probe for the int8-image kernel's operand path: every workgroup (one per CU) streams an L2-resident region
// into LDS with the same LDS-direct buffer loads the kernel's loader waves use, 96 KiB in flight per CU (the kernel's
// three stages), all CUs at once.  Nothing reads the LDS copy; the figure is what the path from L2 through the CU's
// vector memory unit into LDS delivers -- with kWaves issuing waves of kSlots loads in flight each, in contiguous
// 1 KiB pieces or (kRows) in the kernel's own pieces of 8 rows x 128 bytes out of 128 rows.
constexpr int kProbeLdsWaves = 8, kProbeLdsSlots = 12;
template <int kWaves, int kSlots, bool kRows>
__global__ __launch_bounds__(kWaves * 64) void probe_l2_lds_kernel(const unsigned char* __restrict__ buf,
                                                                   size_t region_bytes, int regions, int passes) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const bsi_rsrc r = make_rsrc(buf + static_cast<size_t>(blockIdx.x % regions) * region_bytes, region_bytes);
    const int pieces = static_cast<int>(region_bytes / 1024);
    // kRows: the region is 128 rows of region_bytes / 128 bytes; a piece is 8 rows x 128 bytes (the kernel's stage loads)
    const uint32_t rowbytes = static_cast<uint32_t>(region_bytes / 128);
    const uint32_t lane_off = kRows ? static_cast<uint32_t>(lane >> 3) * rowbytes + static_cast<uint32_t>(lane & 7) * 16
                                    : static_cast<uint32_t>(lane) * 16;
    int slot = 0;
    for (int pass = 0; pass < passes; ++pass)
        for (int p = wave; p < pieces; p += kWaves) {
            const uint32_t wave_off = kRows ? static_cast<uint32_t>(p & 15) * 8 * rowbytes + static_cast<uint32_t>(p >> 4) * 128
                                            : static_cast<uint32_t>(p) * 1024;
            load16_to_lds(r, lane_off, wave_off, lds + (wave * kSlots + slot) * 1024);
            slot = (slot + 1 == kSlots) ? 0 : slot + 1;
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kSlots - 1) : "memory");
        }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// Tile configuration: TM keys x TN queries per workgroup (128 x 128, 128 x 64, 64 x 64 or 64 x 32; the smaller
// ones for grids that would leave CUs without a workgroup), MFMA waves arranged 2 (keys) x kWavesN (queries),
// each WM x WN tiles of 16 x 16; one loader wave per (up to) 64 operand rows.

#ifndef BSI_I8_WN_RULE
#define BSI_I8_WN_RULE ((TM == 128 && TN == 128) ? 2 : 1)
#endif
template <int TM, int TN>
struct I8Cfg {
    static constexpr int kTM = TM, kTN = TN;
    static constexpr int kWM = TM / 32;                // 16-key tiles per wave (2 waves along the keys)
    // 16-query tiles per wave: two for the 128 x 128 tile (eight MFMA waves of 64 x 32), one for the smaller tiles, which
    // would otherwise run on four MFMA waves or fewer -- one per SIMD, and a single wave cannot issue its MFMAs, the chain
    // and the operand reads fast enough to keep its SIMD's matrix pipe busy
    static constexpr int kWN = BSI_I8_WN_RULE;
    static constexpr int kWavesN = TN / (16 * kWN);    // waves along the queries
    static constexpr int kConsumers = 2 * kWavesN;
    static constexpr int kGroups = (TM + TN) / 8;      // groups of 8 operand rows (1 KiB per half-chunk) in a stage
    // loader waves: one per SIMD (the more waves issue a stage's loads, the faster it comes) -- but two for the
    // 64 x 64 tile, measured: on one machine 512 x 8192 x 2048 takes 17.4 us with two and 18.7 with four (with four
    // or with eight MFMA waves alike), while the 64 x 32 and 128 x 64 tiles gain 5 to 10 % from four
    static constexpr int kLoaders = (TM == 64 && TN == 64) ? 2 : 4;
    static constexpr int kLoads = (kGroups + kLoaders - 1) / kLoaders;  // loads per loader wave and stage
    static constexpr int kBlock = (kConsumers + kLoaders) * 64;
    static constexpr int kOperandK = TM * 128;         // bytes of the key tile of one half-chunk
    static constexpr int kStage = (TM + TN) * 128;     // keys then queries
    // chunk scales: a ring of four groups of one or four chunks (i8_scale_shift), [query][chunk of the group] floats
    static constexpr int kScaleRegions = TN >= 64 ? TN / 64 : 1;      // of 64 queries
    static constexpr int kScaleGroup = kScaleRegions * 64 * 4 * 4;    // bytes
    static constexpr int kScaleBytes = 4 * kScaleGroup;
    static constexpr int kEpilogueBytes = 2 * TM * 4;  // the tile's key factors, then its biases (chain modes)
    static constexpr int kLds = 4 * kStage + kScaleBytes + kEpilogueBytes;
    // D-split launches: one flag word per MFMA wave (a prefix of its chain came near the exactness limit), then the
    // workgroup's decision (kSplitLeave / kSplitCombine / kSplitRedo)
    static constexpr int kSplitFlagBytes = 64;
    static constexpr int kLdsSplit = kLds + kSplitFlagBytes;
    static_assert(kConsumers < 15, "flag words of the MFMA waves, then the decision word");
};
constexpr int kSplitLeave = 0, kSplitCombine = 1, kSplitRedo = 2;

// How the chunk scales are fetched (kFour of the kernels): one float of each of 64 queries for every chunk, or four consecutive
// floats of 16 queries, for the group of four chunks after the one a load is issued in.  The scales of a query are contiguous:
// one float of 64 queries is up to 64 lines, half as many again as the operands of a chunk of the 64 x 64 tile have, four floats
// of 16 are 16.  Rows of fewer than 16 chunks have several queries in a line and gain nothing for the code and the loads ahead
// of the first group; nor do row scales.
// us, one and four (64 x 64 tiles) 512 x 8192 x 2048 16.4, 15.5; 256 x 8192 x 1024 11.4, 10.5; (128 x 64) 512 x 4096 x 4096 12.5,
// 11.7; (128 x 128) 512 x 8192 x 8192 34.5, 32.8 -- and at 8 chunks 512 x 2048 x 8192 11.2, 11.5, 512 x 2048 x 2048 5.8, 6.0.
static bool i8_four_scales(int qscale_stride) { return qscale_stride >= 16; }

// Timeline build (make TIMELINE=1, -DBSI_TIMELINE): one MFMA wave and one loader wave of every workgroup of
// dot_mfma_i8_kernel stamp the 100 MHz wall clock at the points below, 8 slots per workgroup (the first
// kTimelineWorkgroups of the grid); bsi_hip_timeline_read copies them out.  The ordinary build has none of this.
constexpr int kTimelineWorkgroups = 8192;
enum TimelineStamp {
    kStampMfmaEntry = 0, kStampFirstStage = 1, kStampLoopDone = 2, kStampStored = 3, kStampLoaderEntry = 4,
    kStampLoaderDone = 5, kStampFirstIssue = 6, kStampThreeIssued = 7
};
#ifdef BSI_TIMELINE
__device__ unsigned long long g_timeline[kTimelineWorkgroups * 8];
__device__ unsigned long long g_timeline_cycles[kTimelineWorkgroups * 8];  // the shader-clock counter at the same points
#define BSI_STAMP(slot)                                                                    \
    {                                                                                      \
        const unsigned wg_ = (blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x; \
        if (lane == 0 && wg_ < kTimelineWorkgroups) {                                      \
            g_timeline[wg_ * 8 + (slot)] = wall_clock64();                                 \
            g_timeline_cycles[wg_ * 8 + (slot)] = clock64();                               \
        }                                                                                  \
    }
#else
#define BSI_STAMP(slot)
#endif

// A loader wave's share of a region that the next dot will read: one lane per 128-byte line, 64 lines per load.  The values
// are summed only so that the loads stay; the store never happens.  The lines are shared among the workgroups that come here: all of the
// grid, or, tiles != 0, those that have a tile (number `tile` of `tiles`; the others of a launch with the build inside, coop_groups, leave
// before).  us a layer of 400 MB of linked layers, unlinked, with the lines shared among the whole grid of such launches, and so: 64 x
// 768 x 768 6.5, 6.7, 6.4; 128 x 768 x 768 6.9, 7.1, 6.8; 256 x 768 x 768 8.1, 8.4, 8.1; 128 x 1024 x 1024 8.1, 8.3, 7.9.
template <int kLoaders>
__device__ __forceinline__ void i8_warm_lines(unsigned char* __restrict__ unused_lds, int lw, int lane, const unsigned char* __restrict__ warm,
                                              long long warm_lines, int tile = 0, int tiles = 0) {
    const long long groups = tiles != 0 ? tiles : static_cast<long long>(gridDim.x) * gridDim.y * gridDim.z;
    const long long group = tiles != 0 ? tile : (static_cast<long long>(blockIdx.z) * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
    const long long waves = groups * kLoaders, mine = group * kLoaders + lw;
    const long long per = (warm_lines + waves - 1) / waves;
    const long long first = mine * per;
    const long long last = (first + per < warm_lines) ? first + per : warm_lines;
    unsigned sum = 0;
    for (long long l = first + lane; l < last; l += 64) sum += *reinterpret_cast<const volatile unsigned*>(warm + l * 128);
    if (sum == 0x5ca1ab1eu && warm_lines < 0) unused_lds[lane] = 0;
}

// A loader wave of the int8-image kernels (lw = its number among the C::kLoaders loader waves; `consumers` MFMA
// waves share the workgroup's barriers with it): 8 of the stage's groups of 8 rows (the TM key rows, then the TN
// query rows: a load moves 1 KiB = 8 rows x 128 bytes), plus the chunk scales of 64 queries once per chunk.
template <typename C, bool kSum, bool kFour>
__device__ __forceinline__ void i8_loader_wave(unsigned char* __restrict__ lds, int lw, int lane,
                                               const int8_t* __restrict__ A8, const float* __restrict__ qscale,
                                               int qscale_stride, const int8_t* __restrict__ K8,
                                               const float* __restrict__ Bw, int Sb, int chunks, int first_chunk,
                                               int halves, int64_t R, int64_t Q, int64_t r0, int64_t q0, size_t rowbytes,
                                               const float* __restrict__ bias, int ndig, long long dig_stride,
                                               int key_tiled, const unsigned char* __restrict__ warm,
                                               long long warm_lines, int tile = 0, int tiles = 0) {
    constexpr int TM = C::kTM, TN = C::kTN;
    constexpr int L = C::kLoaders, NI = C::kLoads, KG = TM / 8, QG = TN / 8;
    // The key groups and the query groups both divide evenly among the loader waves: every loader moves KG / L key
    // groups, then QG / L query groups, so which operand a load belongs to is known at compile time.
    static_assert(KG % L == 0 && QG % L == 0 && NI == KG / L + QG / L, "loads per loader wave");
    unsigned char* const scale_lds = lds + 4 * C::kStage;
    // The prologue below is kept short on purpose: it runs on one wave per SIMD while the whole workgroup waits for
    // the first stage.  No row is clamped: the offset of a lane's ROW (group and row inside it) travels in the
    // per-lane offset of the buffer load, which the hardware compares with the descriptor's size, so a row past its
    // operand's end reads nothing; whatever such a row or query leaves in LDS only reaches outputs past R or Q, which
    // are never stored.  The wave-uniform offset of the load carries the position INSIDE the row only (the
    // half-chunk), so nothing depends on whether that offset takes part in the range check.
    // tiled keys: blocks of 64 rows x 128 bytes per half-chunk, 2 chunks of them per 64-row tile; rows past R
    // are zero padding inside the last block
    const uint32_t rowbytes32 = static_cast<uint32_t>(chunks) << 8;
    const uint32_t kblock = static_cast<uint32_t>(chunks) << 14;  // bytes of a 64-row tile of the tiled image
    const bsi_rsrc rk = key_tiled ? make_rsrc(K8 + static_cast<size_t>(r0 / 64) * kblock,
                                              static_cast<size_t>((R + 63) / 64 - r0 / 64) * kblock)
                                  : make_rsrc(K8 + static_cast<size_t>(r0) * rowbytes,
                                              static_cast<size_t>(R - r0) * rowbytes);
    const bsi_rsrc rq = make_rsrc(A8 + static_cast<size_t>(q0) * rowbytes,
                                  static_cast<size_t>(Q - q0) * rowbytes +
                                      (kSum ? static_cast<size_t>(ndig - 1) * static_cast<size_t>(dig_stride) : 0));
    // A load moves group g of the stage: 8 rows x 128 bytes; lane = (row lr of the group, 16-byte column lc), and the
    // logical column that lands in LDS column lc of row 8 g + lr is lc ^ (((8 g + lr) >> 1) & 7) = lc ^ (4 (g & 1) +
    // (lr >> 1)).  Per lane: the offset inside the group, for either parity of g and for either layout; per load
    // the offset of its group.
    const uint32_t lr = static_cast<uint32_t>(lane) >> 3, lc = static_cast<uint32_t>(lane) & 7;
    uint32_t voff[NI];
    bool is_key[NI];  // known at compile time once the loops are unrolled
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        is_key[i] = i < KG / L;
        const int gg = is_key[i] ? lw + L * i : lw + L * (i - KG / L);  // group of its operand
        const uint32_t col = (lc ^ (static_cast<uint32_t>(gg & 1) * 4 + (lr >> 1))) * 16;
        const bool tiled = is_key[i] && key_tiled;
        voff[i] = (tiled ? lr * 128 : lr * rowbytes32) + col +
                  (tiled ? static_cast<uint32_t>(gg >> 3) * kblock + static_cast<uint32_t>(gg & 7) * 1024
                         : static_cast<uint32_t>(gg) * 8 * rowbytes32);
    }
    const uint32_t kstep_bytes = key_tiled ? 8192u : 128u;  // from one half-chunk of a key row to the next
    // Scales: a load takes those of 1 << sh chunks and 64 >> sh queries, lane = (query, chunk).  One chunk at a time, behind the second half of every chunk, its scales of the 64 queries of this wave's region; in groups of four, behind
    // chunk c, the quarter c % 4 of those queries' for the group after the one c is in.  Waves of a region load the same.  The
    // position inside the row travels in the per-lane offset: what a group has past the end of the last row is not read.
    const bsi_rsrc rs = make_rsrc(qscale + q0 * qscale_stride, static_cast<size_t>(Q - q0) * qscale_stride * 4);
    constexpr int sh = kFour ? 2 : 0;
    const int sstep = (qscale_stride == 1) ? 0 : 4, region = lw % C::kScaleRegions;
    const int soff = (region * 64 + (lane >> sh)) * qscale_stride * 4 + ((lane & ((1 << sh) - 1)) + first_chunk) * sstep;
    auto load_scales = [&](int group, int quarter) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, BSI_LDS_PTR(scale_lds + (group & 3) * C::kScaleGroup + region * 1024 + quarter * 256), 4,
                                                 soff + (quarter * 64 * qscale_stride + (group << sh) * sstep), 0, 0, 0);
    };
    // issue() is called for h = 0, 1, 2, ... in order, h counted from the first half of chunk first_chunk (the
    // workgroup's share of the row in a D-split launch, else 0); in the sum mode (next_c, next_dg) follow the chunk
    // and the digit (counted from the top one) of the half-chunk to come
    int next_c = 0, next_dg = 0;
    uint32_t so_k = 0, so_q = 0;
    auto issue = [&](int h) {  // stage of half-chunk h (clamped to the last) into its ring slot
        const int hc = h < halves ? h : halves - 1;
        if (kSum) {
            if (h < halves) {
                const uint32_t half = static_cast<uint32_t>(next_c) * 2 + static_cast<uint32_t>(h & 1);
                so_k = half * kstep_bytes;
                so_q = half * 128 + static_cast<uint32_t>(ndig - 1 - next_dg) * static_cast<uint32_t>(dig_stride);
                if (h & 1) {
                    if (++next_c == chunks) {
                        next_c = 0;
                        ++next_dg;
                    }
                }
            }
        } else {
            so_q = static_cast<uint32_t>(hc + 2 * first_chunk) * 128;
            so_k = static_cast<uint32_t>(hc + 2 * first_chunk) * kstep_bytes;
        }
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int g = i < KG / L ? lw + L * i : KG + lw + L * (i - KG / L);  // group of the stage
            load16_to_lds(is_key[i] ? rk : rq, voff[i], is_key[i] ? so_k : so_q,
                          lds + (h & 3) * C::kStage + g * 1024);
        }
        if (!kSum && (h & 1)) load_scales(kFour ? (hc >> 3) + 1 : hc >> 1, kFour ? (hc >> 1) & 3 : 0);
    };
    if (lw == 0) BSI_STAMP(kStampFirstIssue);
    issue(0);
    issue(1);
    constexpr int kSharing = L / C::kScaleRegions;  // waves of a region: of a first group of four chunks each loads its part
    constexpr int kFirst = !kSum && kFour ? 4 / kSharing : 0;
#pragma unroll
    for (int k = 0; k < kFirst; ++k) load_scales(0, lw / C::kScaleRegions + kSharing * k);
    issue(2);
    if (lw == 0) BSI_STAMP(kStampThreeIssued);
    // The epilogue's operands, staged once per workgroup behind the first three stages: the slice-0 weight (key
    // factor) and the bias of the tile's TM keys, 64 rows per load.  (Fetched per lane at the end they are 32
    // vector-memory instructions for every MFMA wave, all queued in front of the output stores.)  Every loader wave
    // issues kEpi of them -- wrapping around where they do not divide evenly -- so that the waits below count the
    // same for all.  Rows past R, and the biases of a call without one, read nothing and give 0 (buffer bounds).
    constexpr int kEpi = kSum ? 0 : (2 * (TM / 64) + L - 1) / L;
    if (!kSum) {
        const bsi_rsrc wrs = make_rsrc(Bw + static_cast<size_t>(r0) * Sb, static_cast<size_t>(R - r0) * Sb * sizeof(float));
        const bsi_rsrc brs = make_rsrc(bias != nullptr ? bias + r0 : Bw,
                                       bias != nullptr ? static_cast<size_t>(R - r0) * sizeof(float) : 0);
        unsigned char* const epi = lds + 4 * C::kStage + C::kScaleBytes;
#pragma unroll
        for (int k = 0; k < kEpi; ++k) {
            const int j = (lw + L * k) % (2 * (TM / 64));
            const bool is_bias = j >= TM / 64;
            const int blk = is_bias ? j - TM / 64 : j;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(is_bias ? brs : wrs,
                                                     BSI_LDS_PTR(epi + (is_bias ? TM * 4 : 0) + blk * 256), 4,
                                                     (blk * 64 + lane) * (is_bias ? 4 : Sb * 4), 0, 0, 0);
        }
    }
    // stage 0 landed (stage 1 + scales + stage 2 + the epilogue operands may be in flight)
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NI + (kSum ? 0 : 1) + kFirst + kEpi) : "memory");
    lds_barrier();
    for (int h = 0; h < halves; ++h) {
        if (h + 3 < halves) {
            issue(h + 3);  // its slot was released by the barrier that ended half h - 1
            // stage h + 1 (and the scales issued right behind it) landed; stages h + 2, h + 3 and one
            // scale load, 2 NI + 1 instructions, may still be in flight
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NI + (kSum ? 0 : 1)) : "memory");
        } else if (h + 3 == halves) {
            // nothing left to issue (a copy of the last stage here, as the prologue does for a single chunk, would
            // queue 96 KiB of loads in front of every workgroup's output stores); the last stage and its
            // scales may be in flight
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NI + (kSum ? 0 : 1)) : "memory");
        } else {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        lds_barrier();
    }
    if (warm_lines > 0) i8_warm_lines<L>(scale_lds, lw, lane, warm, warm_lines, tile, tiles);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may still be writing LDS when the workgroup ends
}

// One k-step (64 of a chunk's 256 elements) of an MFMA wave: WM WN MFMAs on the operands in (ka, qb), one
// epilogue element of the previous chunk (held in `prev`) behind each MFMA, and behind the first WM + WN of them
// the reads of the NEXT k-step's operands into (ka_n, qb_n), so that the LDS latency of every k-step hides
// behind the MFMAs of the one before it -- also across the barrier between two stages of the ring.
// KS: k-step of the chunk (0..3); krow_n / qrow_n: the wave's rows of the next k-step's stage, column included.
// kMode: kI8Chain (fp32 chunk-scale chain), kI8Ints (the same, and the per-chunk integers are stored) or kI8Sum
// (plain int32 sum over all chunks: no scales, no epilogue).
constexpr int kI8Chain = 0, kI8Ints = 1, kI8Sum = 2;
#ifndef BSI_SPLIT_TRACK
#define BSI_SPLIT_TRACK kSplit
#endif
template <int WM, int WN, int KS, int kMode, bool kTrack>
__device__ __forceinline__ void i8_kstep(const v4i (&ka)[WM], const v4i (&qb)[WN], v4i (&ka_n)[WM], v4i (&qb_n)[WN],
                                         const unsigned char* __restrict__ krow_n,
                                         const unsigned char* __restrict__ qrow_n, v4i (&acc)[WM][WN],
                                         const v4i (&prev)[WM][WN], float (&accf)[WM][WN][4],
                                         const float (&qs_prev)[WN], int* __restrict__ ints_prev,
                                         const int64_t (&int_off)[WM][WN], const int (&int_rows)[WM], int down_shift,
                                         int chunks, float& peak) {
    // kTrack (D-split launches): `peak` follows the largest magnitude the lane's chain values take, two of them per
    // three-input maximum
    static_assert(WM + WN <= 2 * WM * WN, "two operand reads behind each MFMA of a k-step");
#pragma unroll
    for (int a = 0; a < WM; ++a)
#pragma unroll
        for (int b = 0; b < WN; ++b) {
            const int t = a * WN + b;
            constexpr bool kInts = (kMode == kI8Ints);
            const v4i c0 = (KS == 0 && kMode != kI8Sum) ? (v4i){0, 0, 0, 0} : acc[a][b];
            acc[a][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ka[a], qb[b], c0, 0, 0, 0);
            if (kMode != kI8Sum) {
                const int idx = KS * (WM * WN) + t, tt = idx >> 2, e = idx & 3, ea = tt / WN, eb = tt % WN;
                accf[ea][eb][e] = fmaf(static_cast<float>(prev[ea][eb][e]), qs_prev[eb], accf[ea][eb][e]);
                if (kTrack && (e & 1)) peak = fmaxf(fmaxf(peak, fabsf(accf[ea][eb][e - 1])), fabsf(accf[ea][eb][e]));
                if (kInts && ints_prev != nullptr && int_off[ea][eb] >= 0 && e < int_rows[ea])
                    ints_prev[int_off[ea][eb] + static_cast<int64_t>(e) * chunks] = prev[ea][eb][e] >> down_shift;
            }
            // reads 2 t and 2 t + 1 of the next k-step, in the order its MFMAs first need them: ka[0], qb[0..],
            // ka[1..].  Two per MFMA: the last of them is then issued more than half a k-step before the barrier
            // that may follow this k-step, which has to wait for all of them before it releases their stage.
#pragma unroll
            for (int r = 2 * t; r < 2 * t + 2; ++r) {
                if (r == 0) ka_n[0] = *reinterpret_cast<const v4i*>(krow_n);
                else if (r <= WN) qb_n[r - 1] = *reinterpret_cast<const v4i*>(qrow_n + (r - 1) * 16 * 128);
                else if (r < WM + WN) ka_n[r - WN] = *reinterpret_cast<const v4i*>(krow_n + (r - WN) * 16 * 128);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
}

// The output tile of an MFMA wave (WM x WN tiles of 16 keys x 16 queries; lane (ln, lg) holds keys 4 lg .. + 3 of
// query ln of each) stored in whole 128-byte lines.  Stored as it lies, a store instruction writes 64 bytes per query
// (4 lanes x 16 bytes): half a line.  Here neighbouring query lanes first swap one of two vertically adjacent tiles
// (a, a + 1), so that the even lane holds keys 0 .. 15 of both queries and the odd lane keys 16 .. 31; a store then
// writes, for one query of the pair, 8 lanes x 16 bytes = the 32 consecutive keys of a line.  Queries and keys past the last
// are left out.  An output whose rows do not begin at lines takes the
// same stores (16 bytes at any multiple of 4, which global memory takes; plain ones, since two of them share a line).
// stream_out: nontemporal stores.
// An output of 4801 keys was stored a float a lane before.  us, before and now: 2000 x 1600 x 4801 as a dot 41.6, 27.0, as a layer 48.1,
// 33.1 (4800 keys: 31.7), 512 x 1601 x 4801 17.9, 14.2; 1000 x 1024 x 2046 12.7, 10.7; f16 (i8_store_half) 2000 x 1600 x 4801 46.8, 41.0,
// 1000 x 1024 x 2050 14.3, 11.0.  Tiles that lie inside keep stores without masks (us, with masks in all: 4000 x 512 x 4096 25.1 for 24.2, a
// dot of 1600 x 768 x 4096 12.1 for 11.6); the last keys are stored an output at a time, from the same registers.
template <int WM, int WN>
__device__ __forceinline__ void i8_store_lines(const float (&v)[WM][WN][4], float* __restrict__ out, int64_t R_total,
                                               int64_t rw, int64_t qw, int64_t R, int64_t Q, int ln, int lg,
                                               bool stream_out) {
    static_assert(WM % 2 == 0, "tiles are paired along the keys");
    if ((R_total & 31) != 0 || (reinterpret_cast<uintptr_t>(out) & 127) != 0) stream_out = false;
    const bool odd = (ln & 1) != 0;
    float* const mine = out + (qw + (ln & ~1)) * R_total + rw + (odd ? 16 : 0) + lg * 4;
    typedef float v4f __attribute__((ext_vector_type(4), aligned(4)));
    const auto each = [&](auto put) {
#pragma unroll
        for (int a = 0; a < WM; a += 2)
#pragma unroll
            for (int b = 0; b < WN; ++b) {
                v4f x, y;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float give = odd ? v[a][b][e] : v[a + 1][b][e];
                    // quad_perm [1, 0, 3, 2]: the value of the neighbouring query lane
                    const float got = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(give), 0xB1, 0xF, 0xF, false));
                    x[e] = odd ? got : v[a][b][e];       // the pair's even query: keys 16 (odd lane) + 4 lg ..
                    y[e] = odd ? v[a + 1][b][e] : got;   // the pair's odd query
                }
                put(mine + static_cast<int64_t>(b * 16) * R_total + a * 16, x, y, a, b);
            }
    };
    if (rw + WM * 16 <= R && qw + WN * 16 <= Q) {
        if (stream_out) {  // the output leaves the caches as it is written
            typedef float v4f_aligned __attribute__((ext_vector_type(4)));
            each([&](float* dst, v4f x, v4f y, int, int) {
                __builtin_nontemporal_store(static_cast<v4f_aligned>(x), reinterpret_cast<v4f_aligned*>(dst));
                __builtin_nontemporal_store(static_cast<v4f_aligned>(y), reinterpret_cast<v4f_aligned*>(dst + R_total));
            });
        } else {
            each([&](float* dst, v4f x, v4f y, int, int) {
                *reinterpret_cast<v4f*>(dst) = x;
                *reinterpret_cast<v4f*>(dst + R_total) = y;
            });
        }
        return;
    }
    if (qw >= Q) return;
    each([&](float* dst, v4f x, v4f y, int a, int b) {
        const int64_t queries = Q - (qw + b * 16 + (ln & ~1)), keys = R - (rw + a * 16 + (odd ? 16 : 0) + lg * 4);  // from the lane's first on
        if (rw + WM * 16 <= R) {
            if (queries > 0) *reinterpret_cast<v4f*>(dst) = x;
            if (queries > 1) *reinterpret_cast<v4f*>(dst + R_total) = y;
            return;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (queries > 0 && e < keys) dst[e] = x[e];
            if (queries > 1 && e < keys) dst[R_total + e] = y[e];
        }
    });
}

// The same output tile in a half-precision type (v before the bias; `bi` the biases of the lane's rows).  The lane's four
// keys of a tile are 8 bytes; exchanging one of two vertically adjacent tiles between neighbouring lane rows
// (v_permlane16_swap: odd rows of the first operand with even rows of the second) gives every lane eight consecutive
// keys, so a store instruction writes 64 contiguous bytes per query.
// The type and whether there is a bias are looked at once a call, not once an output: 25 instructions a store where there were 175,
// a branch, two conversions and a choice for each of its eight outputs.  us a layer, before and now: 512 x 2048 x 8192 bf16 17.6, 16.1;
// 1024 x 4096 x 4096 bf16 28.1, 26.8; 4096 x 4096 x 16384 bf16 270, 266, with tiles of 128 x 128 321, 310.  Of 333 x 2048 x 2048 f16 the
// kernel, 7.1, 6.6; the layer is bound by the host, and no faster.
template <int WM, int WN>
__device__ __forceinline__ void i8_store_half(const float (&v)[WM][WN][4], const float (&bi)[WM][4], bool has_bias, int dtype,
                                              float* __restrict__ out, int64_t R_total, int64_t rw, int64_t qw, int64_t R,
                                              int64_t Q, int ln, int lg) {
    unsigned short* const out16 = reinterpret_cast<unsigned short*>(out);
    const bool inside = rw + WM * 16 <= R;
    const auto store = [&](auto type, auto biased) {
        constexpr int kType = decltype(type)::value;
        constexpr bool kBias = decltype(biased)::value;
        float rounded[WM][4];
#pragma unroll
        for (int a = 0; a < WM; ++a)
#pragma unroll
            for (int e = 0; e < 4; ++e) rounded[a][e] = kBias ? half_value(half_bits(bi[a][e], kType), kType) : 0.0f;
#pragma unroll
        for (int a = 0; a < WM; a += 2)
#pragma unroll
            for (int b = 0; b < WN; ++b) {
                uint32_t p[2][2];
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int h = 0; h < 2; ++h)
                        p[t][h] = half_pair<kType, kBias>(v[a + t][b][2 * h], v[a + t][b][2 * h + 1], rounded[a + t][2 * h], rounded[a + t][2 * h + 1]);
                const auto lo = __builtin_amdgcn_permlane16_swap(p[0][0], p[1][0], false, false);
                const auto hi = __builtin_amdgcn_permlane16_swap(p[0][1], p[1][1], false, false);
                const int64_t q = qw + b * 16 + ln, first = rw + (a + (lg & 1)) * 16 + (lg >> 1) * 8;
                typedef uint32_t v4u __attribute__((ext_vector_type(4), aligned(2)));
                const v4u eight = {lo[0], hi[0], lo[1], hi[1]};
                unsigned short* const dst = out16 + static_cast<size_t>(q) * R_total + first;
                if (inside) {
                    if (q < Q) *reinterpret_cast<v4u*>(dst) = eight;
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (q < Q && first + e < R) dst[e] = static_cast<unsigned short>(eight[e >> 1] >> (16 * (e & 1)));
                }
            }
    };
    const auto of_type = [&](auto type) {
        if (has_bias) store(type, std::true_type{});
        else store(type, std::false_type{});
    };
    if (dtype == BSI_DTYPE_F16) of_type(std::integral_constant<int, BSI_DTYPE_F16>{});
    else of_type(std::integral_constant<int, BSI_DTYPE_BF16>{});
}

// The end of a tile in the chain modes: every output takes its key's factor, the decimal scale and the bias, and is stored.
// kHalf: the outputs are in the half-precision type out_dtype, else float32.  One kind of store a kernel: with both in one, a
// launch of a few microseconds fetches instructions it does not run between those it does (us, both and one: 64 x 2048 x 256
// 4.89, 4.77; 40 x 1024 x 1024 3.70, 3.55; 77 x 1600 x 4800 4.63, 4.48; 100 x 1000 x 3000 4.20, 4.03).
// epi: the key factors and biases of the tile's TM rows, from the copy the loader waves staged in LDS (0 for rows past R and
// for a call without bias): two 16-byte reads per 16-key tile.
template <int TM, int WM, int WN, bool kHalf>
__device__ __forceinline__ void i8_store_tile(const float (&accf)[WM][WN][4], const unsigned char* __restrict__ epi_lds, float down,
                                              float scale_inv, bool has_bias, int out_dtype, float* __restrict__ out,
                                              int64_t R_total, int64_t r0, int64_t q0, int wr, int wq, int64_t R, int64_t Q,
                                              int ln, int lg, bool stream_out) {
    const int64_t qw = q0 + wq * (WN * 16);
    const float* epi = reinterpret_cast<const float*>(epi_lds);
#pragma unroll
    for (int a0 = 0; a0 < WM; a0 += 2) {  // two 16-key tiles at a time: what the stores pair up
        const int64_t rw = r0 + wr * (WM * 16) + a0 * 16;
        float v[2][WN][4], bi[2][4];
#pragma unroll
        for (int a = 0; a < 2; ++a) {
            const int rl = wr * (WM * 16) + (a0 + a) * 16 + lg * 4;  // row of the tile
            const float4 w4 = *reinterpret_cast<const float4*>(epi + rl);
            const float4 b4 = *reinterpret_cast<const float4*>(epi + TM + rl);
            const float bs[4] = {key_factor(w4.x), key_factor(w4.y), key_factor(w4.z), key_factor(w4.w)};
            bi[a][0] = b4.x, bi[a][1] = b4.y, bi[a][2] = b4.z, bi[a][3] = b4.w;
#pragma unroll
            for (int b = 0; b < WN; ++b)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    // (acc * key scale) * scale_inv, then + bias: each step rounded on its own, as separate kernels would
                    v[a][b][e] = ((accf[a0 + a][b][e] * down) * bs[e]) * scale_inv;
                    if (!kHalf && has_bias) v[a][b][e] = v[a][b][e] + bi[a][e];
                }
        }
        if constexpr (kHalf) {
            i8_store_half<2, WN>(v, bi, has_bias, out_dtype, out, R_total, rw, qw, R, Q, ln, lg);
            continue;
        }
        i8_store_lines<2, WN>(v, out, R_total, rw, qw, R, Q, ln, lg, stream_out);
    }
}

// Which tile a workgroup takes.  Workgroups go to the eight XCDs in turn, and every XCD has an L2 of its own.  Plain order
// (blockIdx = tile, key tile fastest) gives an XCD the same key tiles in every row of tiles where their number is a multiple
// of 8; elsewhere every XCD came to fetch nearly all keys, once for each query tile.  There, XCD x takes a contiguous run of
// the tiles instead, a key tile at a time through bands of query tiles, so that the workgroups it runs at the same time share
// few key and few query tiles.  us, plain and in bands: 658 x 3840 x 13824 60.4, 49.5; 266 x 2721 x 9017 20.8, 16.6;
// 1500 x 1600 x 6400 32.4, 26.6; 1000 x 4096 x 11008 69.4, 56.6; with whole eighths (2048 x 2048 x 8192) 45.0, 46.1.
struct I8Grid {
    int tiles_x, tiles_y;  // key tiles, query tiles
    int height;            // query tiles of a band (the last may have fewer); 0: plain order
    unsigned by_band, by_height, by_last;  // floor(2^32 / n) + 1 of a band's tiles, its height, the last band's height; 0: n = 1
};
__device__ __forceinline__ unsigned divide_by(unsigned v, unsigned reciprocal) { return reciprocal != 0u ? __umulhi(v, reciprocal) : v; }
__device__ __forceinline__ void i8_tile_of(const I8Grid& g, unsigned id, int& bx, int& by) {
    const unsigned total = static_cast<unsigned>(g.tiles_x) * static_cast<unsigned>(g.tiles_y);
    const unsigned xcd = id & 7u, per = total >> 3, rest = total & 7u;
    const unsigned at = (id >> 3) + xcd * per + (xcd < rest ? xcd : rest);
    const unsigned band = divide_by(at, g.by_band), in = at - band * static_cast<unsigned>(g.tiles_x * g.height);
    const unsigned first = band * static_cast<unsigned>(g.height), left = static_cast<unsigned>(g.tiles_y) - first;
    const bool last = left < static_cast<unsigned>(g.height);
    const unsigned x = divide_by(in, last ? g.by_last : g.by_height);
    bx = static_cast<int>(x);
    by = static_cast<int>(first + in - x * (last ? left : static_cast<unsigned>(g.height)));
}

// The grid of so many of its query tiles.
__device__ __forceinline__ void narrow_grid(I8Grid& g, int tiles_y) {
    g.tiles_y = tiles_y;
    if (g.height == 0) return;
    const unsigned last = static_cast<unsigned>(tiles_y - (tiles_y - 1) / g.height * g.height);
    g.by_last = last == 1u ? 0u : 0xFFFFFFFFu / last + 1u;
}

constexpr int kParts = 3;
template <int TM, int TN, int kMode, bool kSplit, int kBuild, bool kFour, bool kHalf>
__global__ __launch_bounds__((I8Cfg<TM, TN>::kBlock)) void dot_mfma_i8_kernel(
    const int8_t* A8, const float* qscale, int qscale_stride,
    const int8_t* __restrict__ K8,  // int8 key image [R, chunks * 256]
    const float* __restrict__ Bw, int Sb, int chunks, int64_t R, int64_t Q, int down_shift, float scale_inv,
    int64_t R_total, float* __restrict__ out, int* __restrict__ chunk_ints, const float* __restrict__ bias,
    int ndig, long long dig_stride, const long long* __restrict__ key_indices, int key_tiled,
    const unsigned char* __restrict__ warm, long long warm_lines, int out_stream, float* __restrict__ split_partials,
    unsigned* __restrict__ split_counters, float split_limit, int split_shape, I8Grid plain_grid, int out_dtype, CoopBuild coop) {
    // kBuild: the queries are quantised by this launch (bsi_coop_build.h; 1: a chunk a wave at a time, 2: a row); A8 and qscale are
    // not looked at.  kParts (in its place, since it excludes it): the workgroups take parts of the 128 x 128 tiles that split_shape names
    // (launch_mfma_i8_rest); instances of their own, since the others start 0.1 to 0.2 us later with it.
    // kSplit (chain mode only): a D-split launch.  gridDim.z workgroups share an output tile, each running the chain
    // over its own run of chunks from zero.  All operands of the chain are integers (times one power of two), so
    // as long as no value the chain takes exceeds 2^24 of its unit nothing is ever rounded, the value after every
    // chunk is the exact sum so far, and sums of the segments' results in any order equal the one sequential chain over
    // all chunks bit for bit.  Each workgroup follows the largest magnitude its chain values take; with every
    // segment's peak at most split_limit = 2^24 units / gridDim.z, every prefix of the sequential chain is at most
    // 2^24 units as well, which proves the equality.  A workgroup stores its partial sums to split_partials, then
    // counts itself in at split_counters[tile] (bit 16 and up: segments whose peak went over the limit); the last
    // one to arrive adds the others' sums to its own and writes the outputs -- or, if any segment went over the
    // limit, runs the whole tile again over all chunks in order.  It leaves the counter at zero.
    // out_stream: the float outputs of whole tiles go out with nontemporal stores (they leave the caches as they are
    // written) instead of plain ones (they stay for the kernel that reads them next).
    // warm / warm_lines: an optional region of 128-byte lines (the keys the NEXT dot will read) that the loader
    // waves touch once they have issued their last stage, so that it sits in the memory-side cache by the time
    // that dot runs.  (Issued any earlier, from any wave, these long misses hold up the stage loads queued behind
    // them in the CU's vector memory path: measured 40 % slower.)
    // key_tiled: K8 is the tiled image [ceil(R / 64)][2 chunks][64 rows][128 bytes] (a workgroup's key rows of one
    // half-chunk are contiguous, so cold keys stream from HBM in whole pages) instead of row-major [R][chunks * 256].
    // kI8Sum only: A8 holds ndig digit images of the queries, dig_stride bytes apart, lowest digit first; the
    // chunk loop runs over them from the top digit down and the accumulators are shifted left by 7 between two
    // digits (Horner), so that they end as sum_d (sum_i digit_i[q, d] 128^i) K8[r, d].  With chunk_ints the int32
    // sums are stored there ([Q, R_total]); without, out[q, idx[r]] = float(sum * 2^-down_shift * qscale[q *
    // qscale_stride] * Bw[r * Sb]) * scale_inv (+ bias[r]), the product formed in float64.
    using C = I8Cfg<TM, TN>;
    constexpr int WM = C::kWM, WN = C::kWN;
    constexpr bool kInts = (kMode == kI8Ints), kSum = (kMode == kI8Sum);
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];  // C::kLds
    // Which tile, and the first loads' arguments, worked out ahead of the build and held over it: behind it each would be a fetch that all waves
    // wait for.  us, fetched with a branch for workgroups without a tile, and held: 128 x 1024 x 4096 7.5, 7.2; 64 x 960 x 4000 6.8, 6.5.
    [[maybe_unused]] int built_x = static_cast<int>(blockIdx.x), built_y = static_cast<int>(blockIdx.y);
    if constexpr (kBuild == 1 || kBuild == 2) {
        if (plain_grid.height != 0) {
            const int tiles = plain_grid.tiles_x * plain_grid.tiles_y;
            if (built_x < tiles) i8_tile_of(plain_grid, blockIdx.x, built_x, built_y);
            else built_y = plain_grid.tiles_y;
        }
        if (built_y >= plain_grid.tiles_y) built_y = -1;
        asm volatile("" : "+s"(built_x), "+s"(built_y), "+s"(K8), "+s"(chunks), "+s"(Q), "+s"(R));
        coop_build<false, kBuild == 2>(coop, blockIdx.y * gridDim.x + blockIdx.x, reinterpret_cast<unsigned*>(lds), A8, qscale, [] {});
        if (built_y < 0) return;  // there for the build (coop_groups)
    }

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // Which tile (and, in a D-split launch, which segment) this workgroup computes.  A D-split launch is a 1-D grid:
    // key tile fastest, then query tile, then segment, so that workgroups which share a key tile and a run of chunks
    // are neighbours (a grid that gave every XCD one segment of a few key tiles was measured and is no faster).
    int bx, by, seg = 0, nseg = 1, tiles_x = 0;
    if (kSplit) {
        tiles_x = split_shape & 1023;
        const int tiles_y = (split_shape >> 10) & 1023;
        nseg = split_shape >> 20;
        const int id = static_cast<int>(blockIdx.x);
        bx = id % tiles_x;
        by = (id / tiles_x) % tiles_y;
        seg = id / (tiles_x * tiles_y);
    } else {
        bx = static_cast<int>(blockIdx.x), by = static_cast<int>(blockIdx.y);
        if constexpr (kBuild == 1 || kBuild == 2) {
            bx = built_x, by = built_y;
        } else if constexpr (kBuild == kParts) {  // a part past the last key or query does the first one's work
            constexpr int kAcross = 128 / TM;
            const unsigned rest = static_cast<unsigned>(split_shape) & 255u;
            unsigned id = blockIdx.x, part = 0u;
            while (id >= rest) id -= rest, ++part;
            id += static_cast<unsigned>(split_shape) >> 8;
            if (plain_grid.height != 0) {
                i8_tile_of(plain_grid, id, bx, by);
            } else {
                by = static_cast<int>(id / static_cast<unsigned>(plain_grid.tiles_x));
                bx = static_cast<int>(id) - by * plain_grid.tiles_x;
            }
            bx = bx * kAcross + static_cast<int>(part % kAcross);
            by = by * (128 / TN) + static_cast<int>(part / kAcross);
            if (static_cast<int64_t>(bx) * TM >= R) --bx;
            if (static_cast<int64_t>(by) * TN >= Q) --by;
        } else if (plain_grid.height != 0) {
            i8_tile_of(plain_grid, blockIdx.x, bx, by);
        }
    }
    const int64_t r0 = static_cast<int64_t>(bx) * TM;
    const int64_t q0 = static_cast<int64_t>(by) * TN;
    const size_t rowbytes = static_cast<size_t>(chunks) * 256;
    static_assert(!kSplit || kMode == kI8Chain, "only the plain chain splits D");
    const int vchunks = kSum ? chunks * ndig : chunks;  // chunks of the loop: every digit image runs over all chunks
    // the workgroup's run of chunks: all of them, or segment seg of nseg
    const int first_chunk = kSplit ? (chunks * seg) / nseg : 0;
    const int my_chunks = kSplit ? (chunks * (seg + 1)) / nseg - first_chunk : vchunks;
    unsigned char* const scale_lds = lds + 4 * C::kStage;
    // kSplit: [MFMA wave] flags, [15] = decision
    volatile __attribute__((address_space(3))) int* const split_flags =
        reinterpret_cast<volatile __attribute__((address_space(3))) int*>(BSI_LDS_PTR(lds + C::kLds));

    if (wave >= C::kConsumers) {
        if (wave == C::kConsumers) BSI_STAMP(kStampLoaderEntry);
        constexpr bool kHelpers = kBuild == 1 || kBuild == 2;  // workgroups beyond the tiles do not come here
        i8_loader_wave<C, kSum, kFour>(lds, wave - C::kConsumers, lane, A8, qscale, qscale_stride, K8, Bw, Sb, chunks, first_chunk,
                                my_chunks * 2, R, Q, r0, q0, rowbytes, bias, ndig, dig_stride, key_tiled, warm, warm_lines,
                                kHelpers ? by * plain_grid.tiles_x + bx : 0, kHelpers ? plain_grid.tiles_x * plain_grid.tiles_y : 0);
        if (kSplit) {
            lds_barrier();  // the MFMA waves have stored their partial sums
            lds_barrier();  // the decision is in LDS
            if (__builtin_amdgcn_readfirstlane(split_flags[15]) == kSplitRedo)
                i8_loader_wave<C, kSum, kFour>(lds, wave - C::kConsumers, lane, A8, qscale, qscale_stride, K8, Bw, Sb, chunks, 0,
                                        chunks * 2, R, Q, r0, q0, rowbytes, bias, ndig, dig_stride, key_tiled, nullptr, 0);
        }
        if (wave == C::kConsumers) BSI_STAMP(kStampLoaderDone);
        return;
    }
    if (wave == 0) BSI_STAMP(kStampMfmaEntry);

    // ---- MFMA waves
    const int wr = wave & 1, wq = wave >> 1;  // half of the keys, group of 32 queries
    const int ln = lane & 15, lg = lane >> 4;
    const int krow_off = (wr * (WM * 16) + ln) * 128;
    const int qrow_off = C::kOperandK + (wq * (WN * 16) + ln) * 128;
    int pcol[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) pcol[kk] = ((kk * 4 + lg) ^ (ln >> 1)) * 16;
    float accf[WM][WN][4];
#pragma unroll
    for (int a = 0; a < WM; ++a)
#pragma unroll
        for (int b = 0; b < WN; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) accf[a][b][e] = 0.0f;
    v4i acc0[WM][WN], acc1[WM][WN];
#pragma unroll
    for (int a = 0; a < WM; ++a)
#pragma unroll
        for (int b = 0; b < WN; ++b) acc0[a][b] = acc1[a][b] = (v4i){0, 0, 0, 0};
    // the MFMA accumulators hold 2^down_shift times the integer dot; the chain runs on them unscaled
    // (a power of two commutes with every rounding) and the factor is taken out once at the end
    const float down = __uint_as_float(static_cast<uint32_t>(127 - down_shift) << 23);
    int64_t int_off[WM][WN];
    int int_rows[WM];
#pragma unroll
    for (int a = 0; a < WM; ++a) {
        const int64_t r = r0 + wr * (WM * 16) + a * 16 + lg * 4;
        int_rows[a] = static_cast<int>((R - r) < 4 ? (R - r) : 4);
#pragma unroll
        for (int b = 0; b < WN; ++b) {
            const int64_t q = q0 + wq * (WN * 16) + b * 16 + ln;
            int_off[a][b] = (kInts && q < Q && r < R) ? (q * R + r) * chunks : -1;
        }
    }
    // chunk scales of the lane's query columns, from the loaders' ring
    constexpr int sh = kFour ? 2 : 0;
    const int qfirst = wq * (WN * 16);
    const unsigned char* sread = scale_lds + (qfirst >> 6) * 1024 + (((qfirst & 63) + ln) << (2 + sh));
    float qsa[WN], qsb[WN];  // scales of even / odd chunks
#pragma unroll
    for (int b = 0; b < WN; ++b) qsa[b] = qsb[b] = 0.0f;
#define BSI_I8_SCALES(dst, c)                                                                                  \
    {                                                                                                          \
        _Pragma("unroll") for (int b = 0; b < WN; ++b) dst[b] =                                                \
            *reinterpret_cast<const float*>(sread + ((c) >> sh & 3) * C::kScaleGroup + ((c) & ((1 << sh) - 1)) * 4 + (b * 64 << sh)); \
    }
    // The k-steps run one behind their operand reads: k-step j's MFMAs cover the reads of k-step j + 1.  A
    // stage (half-chunk, two k-steps) is released to the loaders by the barrier that follows the k-step in
    // which its last operands were read (the even ones); the same barrier tells that the next stage has landed.
    v4i ka[2][WM], qb[2][WN];  // operand sets of even / odd k-steps
#define BSI_I8_KSTEP(KS, nslot, acc, prev, qs, ip)                                                                  \
    i8_kstep<WM, WN, KS, kMode, BSI_SPLIT_TRACK>(ka[(KS) & 1], qb[(KS) & 1], ka[((KS) + 1) & 1], qb[((KS) + 1) & 1],         \
                                lds + (nslot) * C::kStage + krow_off + pcol[((KS) + 1) & 1],                        \
                                lds + (nslot) * C::kStage + qrow_off + pcol[((KS) + 1) & 1], acc, prev, accf, qs,   \
                                ip, int_off, int_rows, down_shift, chunks, peak);
    // a chunk whose halves sit in ring slots s0, s0 + 1; nslot: slot of the next chunk's first half
#define BSI_I8_CHUNK(s0, nslot, acc, prev, qs, ip)                                                                  \
    BSI_I8_KSTEP(0, s0, acc, prev, qs, ip);                                                                         \
    lds_barrier();                                                                                                  \
    BSI_I8_KSTEP(1, (s0) + 1, acc, prev, qs, ip);                                                                   \
    BSI_I8_KSTEP(2, (s0) + 1, acc, prev, qs, ip);                                                                   \
    lds_barrier();                                                                                                  \
    BSI_I8_KSTEP(3, nslot, acc, prev, qs, ip);

    float peak = 0.0f;      // kSplit: the largest magnitude the lane's chain values have taken
    int run_chunks = my_chunks;
    bool last_in_acc0 = false;
#pragma nounroll
    for (int pass = 0;; ++pass) {  // one pass; a D-split launch's last workgroup of a tile may need a second over all chunks
    if (kSplit && pass > 0) {
#pragma unroll
        for (int a = 0; a < WM; ++a)
#pragma unroll
            for (int b = 0; b < WN; ++b) {
                acc0[a][b] = acc1[a][b] = (v4i){0, 0, 0, 0};
#pragma unroll
                for (int e = 0; e < 4; ++e) accf[a][b][e] = 0.0f;
            }
#pragma unroll
        for (int b = 0; b < WN; ++b) qsa[b] = qsb[b] = 0.0f;
    }
    lds_barrier();  // stage 0 is there
    if (wave == 0) BSI_STAMP(kStampFirstStage);
#pragma unroll
    for (int t = 0; t < WM; ++t) ka[0][t] = *reinterpret_cast<const v4i*>(lds + krow_off + t * 16 * 128 + pcol[0]);
#pragma unroll
    for (int t = 0; t < WN; ++t) qb[0][t] = *reinterpret_cast<const v4i*>(lds + qrow_off + t * 16 * 128 + pcol[0]);
    __builtin_amdgcn_sched_barrier(0);
    // sum mode: before the first chunk of every digit but the top one, the sums so far move up by one digit
    int to_next_digit = chunks;
#define BSI_I8_HORNER()                                                               \
    if (kSum && ndig > 1) {                                                           \
        if (to_next_digit == 0) {                                                     \
            _Pragma("unroll") for (int a = 0; a < WM; ++a)                            \
                _Pragma("unroll") for (int b = 0; b < WN; ++b)                        \
                    _Pragma("unroll") for (int e = 0; e < 4; ++e) acc0[a][b][e] <<= 7; \
            to_next_digit = chunks;                                                   \
        }                                                                             \
        --to_next_digit;                                                              \
    }
    int c = 0;
    for (; c + 1 < run_chunks; c += 2) {
        int* const ip = (!kSum && c > 0) ? chunk_ints + (c - 1) : nullptr;
        // even chunk c -> acc0, ring slots 0 and 1; epilogue of chunk c-1 (acc1, scales qsb)
        BSI_I8_HORNER();
        BSI_I8_CHUNK(0, 2, acc0, acc1, qsb, ip);
        if (!kSum) BSI_I8_SCALES(qsa, c);  // landed with the second half of chunk c
        // odd chunk c+1 -> acc1, ring slots 2 and 3; epilogue of chunk c (acc0, scales qsa)
        if (kSum) {
            BSI_I8_HORNER();
            BSI_I8_CHUNK(2, 0, acc0, acc1, qsb, ip);  // int32 sum: one accumulator set over all chunks
        } else {
            BSI_I8_CHUNK(2, 0, acc1, acc0, qsa, chunk_ints + c);
            BSI_I8_SCALES(qsb, c + 1);
        }
    }
    last_in_acc0 = false;
    if (c < run_chunks) {  // odd number of chunks: one more even chunk; its halves sit in slots 0 and 1
        int* const ip = (!kSum && c > 0) ? chunk_ints + (c - 1) : nullptr;
        BSI_I8_HORNER();
        BSI_I8_CHUNK(0, 2, acc0, acc1, qsb, ip);
        if (!kSum) BSI_I8_SCALES(qsa, c);
        last_in_acc0 = true;
    }
    // the last k-step read ahead into a stage that does not exist (the loaders fill it with a copy of the last
    // one); nothing uses those operands
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (wave == 0) BSI_STAMP(kStampLoopDone);
    if (!kSplit) break;
    if (kSplit) {
        // the chain step of the run's last chunk
#pragma unroll
        for (int a = 0; a < WM; ++a)
#pragma unroll
            for (int b = 0; b < WN; ++b)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int v = last_in_acc0 ? acc0[a][b][e] : acc1[a][b][e];
                    accf[a][b][e] = fmaf(static_cast<float>(v), last_in_acc0 ? qsa[b] : qsb[b], accf[a][b][e]);
                    peak = fmaxf(peak, fabsf(accf[a][b][e]));
                }
        if (pass > 0) break;  // the whole row in order: these are the sequential chain's values
        typedef float v4f __attribute__((ext_vector_type(4)));
        // (formed here, from values the compiler cannot see through, so that no address of the partial sums is
        // computed ahead of the chunk loop and held in registers the loop has none to spare of)
        int lane_late = lane, tile_late = by * tiles_x + bx;
        asm volatile("" : "+v"(lane_late), "+s"(tile_late));
        const size_t tile = static_cast<size_t>(tile_late);
        constexpr size_t kWaveVecs = static_cast<size_t>(WM) * WN * 64;  // 16-byte pieces of an MFMA wave's outputs
        v4f* const parts = reinterpret_cast<v4f*>(split_partials) + tile * nseg * (C::kConsumers * kWaveVecs);
        {
            v4f* mine = parts + (static_cast<size_t>(seg) * C::kConsumers + wave) * kWaveVecs + lane_late;
#pragma unroll
            for (int a = 0; a < WM; ++a)
#pragma unroll
                for (int b = 0; b < WN; ++b)
                    __builtin_nontemporal_store((v4f){accf[a][b][0], accf[a][b][1], accf[a][b][2], accf[a][b][3]},
                                                mine + (a * WN + b) * 64);
        }
        const int wave_over = (__builtin_amdgcn_ballot_w64(!(peak <= split_limit)) != 0) ? 1 : 0;  // any lane of the wave
        if (lane == 0) split_flags[wave] = wave_over;
        // This wave's partial sums have reached the L2 (stores are counted down once the L2 has them).  One lane of
        // the workgroup then makes the whole workgroup's stores visible to the device (a release fence writes back
        // the L2's dirty lines, whichever wave wrote them) before it counts the workgroup in: one write-back per
        // workgroup.  Fences from every wave, and fences that also invalidate, cost the launch ten times the split's gain.
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lds_barrier();
        if (wave == 0 && lane == 0) {
            unsigned any = 0;
            for (int w = 0; w < C::kConsumers; ++w) any |= static_cast<unsigned>(split_flags[w]);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
            const unsigned old = __hip_atomic_fetch_add(split_counters + tile, 1u + (any ? 0x10000u : 0u), __ATOMIC_RELAXED,
                                                        __HIP_MEMORY_SCOPE_AGENT);
            int decision = kSplitLeave;
            if ((old & 0xFFFFu) == static_cast<unsigned>(nseg - 1)) {  // the tile's last workgroup
                // what the other workgroups stored before they counted themselves in, not what this CU's caches
                // may hold of an earlier launch: the invalidation is the CU's, so it serves the waves that load
                // behind the barrier below
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the invalidation has been carried out, not just issued
                decision = ((old >> 16) != 0 || any != 0) ? kSplitRedo : kSplitCombine;
                __hip_atomic_store(split_counters + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next launch
                // running totals behind the tile counters: tiles combined, tiles computed again
                __hip_atomic_fetch_add(split_counters + kSplitMaxTiles + (decision == kSplitRedo ? 1 : 0), 1u,
                                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            split_flags[15] = decision;
        }
        lds_barrier();
        const int decision = __builtin_amdgcn_readfirstlane(split_flags[15]);
        if (decision == kSplitLeave) return;
        if (decision == kSplitCombine) {
            for (int sg = 0; sg < nseg; ++sg) {
                if (sg == seg) continue;
                const v4f* theirs = parts + (static_cast<size_t>(sg) * C::kConsumers + wave) * kWaveVecs + lane_late;
#pragma unroll
                for (int a = 0; a < WM; ++a)
#pragma unroll
                    for (int b = 0; b < WN; ++b) {
                        const v4f v = __builtin_nontemporal_load(theirs + (a * WN + b) * 64);
#pragma unroll
                        for (int e = 0; e < 4; ++e) accf[a][b][e] += v[e];  // exact: see the head of the kernel
                    }
            }
            break;
        }
        run_chunks = chunks;  // kSplitRedo: the loader waves fill the ring from chunk 0 again
    }
    }  // passes
#undef BSI_I8_HORNER
#undef BSI_I8_CHUNK
#undef BSI_I8_KSTEP
#undef BSI_I8_SCALES
    if (kSum && chunk_ints != nullptr) {  // the plain integer sums, int32 [Q, R_total]
#pragma unroll
        for (int a = 0; a < WM; ++a) {
            const int64_t rb = r0 + wr * (WM * 16) + a * 16 + lg * 4;
#pragma unroll
            for (int b = 0; b < WN; ++b) {
                const int64_t q = q0 + wq * (WN * 16) + b * 16 + ln;
                if (q >= Q) continue;
                int* dst = chunk_ints + static_cast<size_t>(q) * R_total + rb;
                if (rb + 3 < R && ((reinterpret_cast<uintptr_t>(dst) & 15) == 0)) {
                    *reinterpret_cast<v4i*>(dst) = acc0[a][b];
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (rb + e < R) dst[e] = acc0[a][b][e];
                }
            }
        }
        return;
    }
    if (kSum) {  // float(sum * 2^-down_shift * query factor * key factor) * scale_inv (+ bias), the product in float64
        const double down2 = __longlong_as_double(static_cast<long long>(1023 - down_shift) << 52);
        double qf[WN];
#pragma unroll
        for (int b = 0; b < WN; ++b) {
            const int64_t q = q0 + wq * (WN * 16) + b * 16 + ln;
            qf[b] = (q < Q) ? static_cast<double>(qscale[q * qscale_stride]) * down2 : 0.0;
        }
        if (key_indices == nullptr) {
            // identity key order: the key factors and biases of all the wave's rows in one round trip (buffer loads:
            // rows past R and a missing bias read nothing and give 0), then four outputs per store
            float kfv[WM][4], biv[WM][4];
            const bsi_rsrc wrs = make_rsrc(Bw, static_cast<size_t>(R) * Sb * sizeof(float));
            const bsi_rsrc brs = make_rsrc(bias != nullptr ? bias : Bw, bias != nullptr ? static_cast<size_t>(R) * sizeof(float) : 0);
#pragma unroll
            for (int a = 0; a < WM; ++a) {
                const int rb = static_cast<int>(r0 + wr * (WM * 16) + a * 16 + lg * 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    kfv[a][e] = __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(wrs, (rb + e) * Sb * 4, 0, 0));
                    biv[a][e] = __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(brs, (rb + e) * 4, 0, 0));
                }
            }
#pragma unroll
            for (int a = 0; a < WM; ++a)
#pragma unroll
                for (int b = 0; b < WN; ++b)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        float v = static_cast<float>(static_cast<double>(acc0[a][b][e]) * qf[b] * static_cast<double>(kfv[a][e])) * scale_inv;
                        if (bias != nullptr) v = v + biv[a][e];
                        accf[a][b][e] = v;
                    }
            i8_store_lines<WM, WN>(accf, out, R_total, r0 + wr * (WM * 16), q0 + wq * (WN * 16), R, Q, ln, lg, out_stream != 0);
            return;
        }
#pragma unroll
        for (int a = 0; a < WM; ++a) {
            const int64_t rb = r0 + wr * (WM * 16) + a * 16 + lg * 4;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int64_t r = rb + e;
                if (r >= R) continue;
                const double kf = static_cast<double>(Bw[r * Sb]);
                const float bi = bias != nullptr ? bias[r] : 0.0f;
                const int64_t col = key_indices ? key_indices[r] : r;
#pragma unroll
                for (int b = 0; b < WN; ++b) {
                    const int64_t q = q0 + wq * (WN * 16) + b * 16 + ln;
                    if (q >= Q) continue;
                    float v = static_cast<float>(static_cast<double>(acc0[a][b][e]) * qf[b] * kf) * scale_inv;
                    if (bias != nullptr) v = v + bi;
                    out[static_cast<size_t>(q) * R_total + col] = v;
                }
            }
        }
        return;
    }
    // epilogue of the last chunk (a D-split launch has done it above)
    if (!kSplit)
#pragma unroll
    for (int a = 0; a < WM; ++a)
#pragma unroll
        for (int b = 0; b < WN; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int v = last_in_acc0 ? acc0[a][b][e] : acc1[a][b][e];
                const float qsv = last_in_acc0 ? qsa[b] : qsb[b];
                accf[a][b][e] = fmaf(static_cast<float>(v), qsv, accf[a][b][e]);
                if (kInts && int_off[a][b] >= 0 && e < int_rows[a])
                    chunk_ints[int_off[a][b] + static_cast<int64_t>(e) * chunks + (chunks - 1)] = v >> down_shift;
            }
    i8_store_tile<TM, WM, WN, kMode == kI8Chain && kHalf>(accf, lds + 4 * C::kStage + C::kScaleBytes, down, scale_inv, bias != nullptr, out_dtype,
                                                 out, R_total, r0, q0, wr, wq, R, Q, ln, lg, out_stream != 0);
#ifdef BSI_TIMELINE
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the stamp below: the outputs have left the wave
    if (wave == 0) BSI_STAMP(kStampStored);
#endif
}

// ------------------------------------------------------------------ int8 image, several tiles a workgroup
//
// Grids of more than one round: one workgroup per CU takes tiles `grid` apart and never drains its ring.  The loader waves go
// on to the next tile's stages while the MFMA waves end one, so of what a workgroup of dot_mfma_i8_kernel spends outside the
// chunk loop (4096 x 4096 x 16384, per tile: 15.0 us of loop, 1.7 to the first stage, 1.7 of stores, 0.9 until the next
// workgroup starts) only the issue of the stores is left.  Same waves, ring, k-steps and chain, so the same bits.
// us before and after: 4096 x 4096 x 16384 312, 294; 2048 x 2048 x 8192 47.1, 43.6; 2772 x 512 x 12800 46.7, 40.2;
// 8192 x 1024 x 4096 58.1, 51.8; 1773 x 5376 x 8704 90.5, 88.3.  What is left at long rows is the chunk loop at the clock the
// chip holds: the launch takes 557 k cycles, 262 k of them with the matrix pipes busy, at 1.9 GHz for the first twenty launches from
// an idle GPU (292 us) and at 1.7 to 1.8 after that (310 to 330); hiding the rest lowers the clock a little further.
template <int TM, int TN>
struct I8TilesCfg : I8Cfg<TM, TN> {
    using C = I8Cfg<TM, TN>;
    static constexpr int kScaleBytes = 4 * C::kLoaders * 256;  // chunk scales: ring of 4 chunks x loader regions x 64 floats
    static constexpr int kLdsTiles = 4 * C::kStage + kScaleBytes + 4 * C::kEpilogueBytes;  // four sets of key factors and biases
};

// The bands of kLargeTile queries that dot_mfma_i8_large_kernel leaves to the chain: their number, then the bands, in ascending order.
// The tiles of that launch are those bands' own, two query tiles a band (one in a last band of half a tile), numbered through as if there were
// no others: left_tile is the query tile of the matrix.
template <bool kLeft>
using LeftBands = std::conditional_t<kLeft, const unsigned*, int>;
__device__ __forceinline__ int left_tile(const unsigned* __restrict__ left, int by) {
    return 2 * static_cast<int>(left[1 + (by >> 1)]) + (by & 1);
}
__device__ __forceinline__ unsigned left_grid(const unsigned* __restrict__ left, I8Grid& g) {  // narrows g to them; the number of tiles
    const int bands = static_cast<int>(left[0]);
    if (bands == 0) return 0u;
    const int half = (g.tiles_y & 1) != 0 && static_cast<int>(left[bands]) == g.tiles_y >> 1 ? 1 : 0;
    narrow_grid(g, 2 * bands - half);
    return static_cast<unsigned>(g.tiles_x) * static_cast<unsigned>(g.tiles_y);
}

// A loader wave: the stages of all the workgroup's tiles, one after the other; three stages ahead of the MFMA waves, across
// the ends of tiles.
template <typename C, bool kLeft>
__device__ __forceinline__ void i8_tiles_loader_wave(unsigned char* __restrict__ lds, int lw, int lane, const int8_t* __restrict__ A8,
                                                     const float* __restrict__ qscale, int qscale_stride,
                                                     const int8_t* __restrict__ K8, const float* __restrict__ Bw, int Sb, int chunks,
                                                     int64_t R, int64_t Q, const float* __restrict__ bias, int key_tiled,
                                                     const I8Grid& grid, unsigned tiles, [[maybe_unused]] LeftBands<kLeft> left) {
    constexpr int TM = C::kTM, TN = C::kTN;
    constexpr int L = C::kLoaders, NI = C::kLoads, KG = TM / 8, QG = TN / 8;
    constexpr int kEpi = (2 * (TM / 64) + L - 1) / L;
    static_assert(KG % L == 0 && QG % L == 0 && NI == KG / L + QG / L, "loads per loader wave");
    const uint32_t rowbytes = static_cast<uint32_t>(chunks) << 8, kblock = static_cast<uint32_t>(chunks) << 14;
    const uint32_t lr = static_cast<uint32_t>(lane) >> 3, lc = static_cast<uint32_t>(lane) & 7;
    uint32_t voff[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const bool is_key = i < KG / L;
        const int gg = is_key ? lw + L * i : lw + L * (i - KG / L);
        const uint32_t col = (lc ^ (static_cast<uint32_t>(gg & 1) * 4 + (lr >> 1))) * 16;
        const bool tiled = is_key && key_tiled;
        voff[i] = (tiled ? lr * 128 : lr * rowbytes) + col +
                  (tiled ? static_cast<uint32_t>(gg >> 3) * kblock + static_cast<uint32_t>(gg & 7) * 1024
                         : static_cast<uint32_t>(gg) * 8 * rowbytes);
    }
    const uint32_t kstep_bytes = key_tiled ? 8192u : 128u;
    const uint32_t soff = static_cast<uint32_t>((lw % (TN >= 64 ? TN / 64 : 1)) * 64 + lane) * static_cast<uint32_t>(qscale_stride) * 4;
    const int sstep = (qscale_stride == 1) ? 0 : 4;
    const int halves = 2 * chunks, epi_at = halves > 2 ? 2 : 1;
    unsigned id = blockIdx.x;       // the tile the next stage belongs to
    int h = 0, ring = 0, tile = 0;  // its half-chunk there, its place in the ring (counted on), the tile's number here
    bsi_rsrc rk, rq, rs, wrs, brs;
    auto enter = [&] {
        int bx, by;
        if (grid.height != 0) {
            i8_tile_of(grid, id, bx, by);
        } else {
            by = static_cast<int>(id / static_cast<unsigned>(grid.tiles_x));
            bx = static_cast<int>(id) - by * grid.tiles_x;
        }
        if constexpr (kLeft) by = left_tile(left, by);
        const int64_t r0 = static_cast<int64_t>(bx) * TM, q0 = static_cast<int64_t>(by) * TN;
        rk = key_tiled ? make_rsrc(K8 + static_cast<size_t>(r0 / 64) * kblock, static_cast<size_t>((R + 63) / 64 - r0 / 64) * kblock)
                       : make_rsrc(K8 + static_cast<size_t>(r0) * rowbytes, static_cast<size_t>(R - r0) * rowbytes);
        rq = make_rsrc(A8 + static_cast<size_t>(q0) * rowbytes, static_cast<size_t>(Q - q0) * rowbytes);
        rs = make_rsrc(qscale + q0 * qscale_stride, static_cast<size_t>(Q - q0) * qscale_stride * 4);
        wrs = make_rsrc(Bw + static_cast<size_t>(r0) * Sb, static_cast<size_t>(R - r0) * Sb * sizeof(float));
        brs = make_rsrc(bias != nullptr ? bias + r0 : Bw, bias != nullptr ? static_cast<size_t>(R - r0) * sizeof(float) : 0);
    };
    enter();
    auto issue = [&] {
        if (h == halves) {
            h = 0;
            id += gridDim.x;
            ++tile;
            enter();
        }
        const uint32_t so_k = static_cast<uint32_t>(h) * kstep_bytes, so_q = static_cast<uint32_t>(h) * 128;
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int g = i < KG / L ? lw + L * i : KG + lw + L * (i - KG / L);
            load16_to_lds(i < KG / L ? rk : rq, voff[i], i < KG / L ? so_k : so_q, lds + (ring & 3) * C::kStage + g * 1024);
        }
        if (h & 1)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rs, BSI_LDS_PTR(lds + 4 * C::kStage + (((ring >> 1) & 3) * L + lw) * 256), 4, static_cast<int>(soff), (h >> 1) * sstep, 0, 0);
        if (h == epi_at) {  // tiles of one chunk: the MFMA waves may still be reading the set of two tiles ago
            unsigned char* const epi = lds + 4 * C::kStage + I8TilesCfg<TM, TN>::kScaleBytes + (tile & 3) * C::kEpilogueBytes;
#pragma unroll
            for (int k = 0; k < kEpi; ++k) {
                const int j = (lw + L * k) % (2 * (TM / 64));
                const bool is_bias = j >= TM / 64;
                const int blk = is_bias ? j - TM / 64 : j;
                __builtin_amdgcn_raw_ptr_buffer_load_lds(is_bias ? brs : wrs, BSI_LDS_PTR(epi + (is_bias ? TM * 4 : 0) + blk * 256), 4,
                                                         (blk * 64 + lane) * (is_bias ? 4 : Sb * 4), 0, 0, 0);
            }
        }
        ++h;
        ++ring;
    };
    const int mine = static_cast<int>((tiles - blockIdx.x + gridDim.x - 1) / gridDim.x), total = mine * halves;
    issue();
    issue();
    if (total > 2) issue();
    // The waits count the loads of the newer stages; the epilogue operands among them only make a wait stricter.
    if (total > 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NI + 1) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();
    for (int g = 0; g < total; ++g) {
        if (g + 3 < total) {
            issue();
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NI + 1) : "memory");
        } else if (g + 3 == total) {
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NI + 1) : "memory");
        } else {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        lds_barrier();
    }
}

template <int TM, int TN, bool kHalf, bool kLeft>
__global__ __launch_bounds__((I8Cfg<TM, TN>::kBlock)) void dot_mfma_i8_tiles_kernel(
    const int8_t* __restrict__ A8, const float* __restrict__ qscale, int qscale_stride, const int8_t* __restrict__ K8,
    const float* __restrict__ Bw, int Sb, int chunks, int64_t R, int64_t Q, int down_shift, float scale_inv, int64_t R_total,
    float* __restrict__ out, const float* __restrict__ bias, int key_tiled, const unsigned char* __restrict__ warm,
    long long warm_lines, int out_stream, I8Grid grid, unsigned tiles, int out_dtype, LeftBands<kLeft> left) {
    // kLeft: the tiles of the bands that dot_mfma_i8_large_kernel, before this launch, has left to it; `grid` is that of all tiles.
    // The keys of the next dot are touched here only if it has left them all (then none of its workgroups has).
    using C = I8Cfg<TM, TN>;
    constexpr int WM = C::kWM, WN = C::kWN, kMode = kI8Chain;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];  // I8TilesCfg::kLdsTiles
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if constexpr (kLeft) {  // the same in all waves of a workgroup
        static_assert(2 * TN == kLargeTile, "two query tiles a band");
        const unsigned all = tiles;
        tiles = left_grid(left, grid);
        if (blockIdx.x >= tiles) return;
        if (tiles != all) warm_lines = 0;
    }
    if (wave >= C::kConsumers) {
        const int lw = wave - C::kConsumers;
        i8_tiles_loader_wave<C, kLeft>(lds, lw, lane, A8, qscale, qscale_stride, K8, Bw, Sb, chunks, R, Q, bias, key_tiled, grid, tiles, left);
        if (warm_lines > 0) i8_warm_lines<C::kLoaders>(lds + 4 * C::kStage, lw, lane, warm, warm_lines);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing may still be writing LDS when the workgroup ends
        return;
    }

    // ---- MFMA waves (see dot_mfma_i8_kernel)
    const int wr = wave & 1, wq = wave >> 1;
    const int ln = lane & 15, lg = lane >> 4;
    const int krow_off = (wr * (WM * 16) + ln) * 128;
    const int qrow_off = C::kOperandK + (wq * (WN * 16) + ln) * 128;
    int pcol[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) pcol[kk] = ((kk * 4 + lg) ^ (ln >> 1)) * 16;
    float accf[WM][WN][4];
    v4i acc0[WM][WN], acc1[WM][WN];
#pragma unroll
    for (int a = 0; a < WM; ++a)
#pragma unroll
        for (int b = 0; b < WN; ++b) {
            acc0[a][b] = acc1[a][b] = (v4i){0, 0, 0, 0};
#pragma unroll
            for (int e = 0; e < 4; ++e) accf[a][b][e] = 0.0f;
        }
    const float down = __uint_as_float(static_cast<uint32_t>(127 - down_shift) << 23);
    const int64_t int_off[WM][WN] = {};
    const int int_rows[WM] = {};
    float peak = 0.0f;
    unsigned char* const scale_lds = lds + 4 * C::kStage;
    const int qfirst = wq * (WN * 16);
    const unsigned char* sread = scale_lds + (qfirst >> 6) * 256 + ((qfirst & 63) + ln) * 4;
    float qsa[WN], qsb[WN];
#pragma unroll
    for (int b = 0; b < WN; ++b) qsa[b] = qsb[b] = 0.0f;
    v4i ka[2][WM], qb[2][WN];
    // the ring's two pairs of slots: the tile's even chunks sit in the pair at `even`, its odd ones in the other
    int even = 0, odd = 2 * C::kStage, chunk0 = 0;
    // A chunk's own scales, which landed with its second half, are read in its middle: the next chunk's first chain step needs them,
    // and read behind the chunk it waited for them (us: 4096 x 4096 x 16384 293 -> 284, 2048 x 2048 x 8192 42.0 -> 40.8; a workgroup
    // of one tile gains nothing by it).
#define BSI_TILES_CHUNK(here, next, acc, prev, qs, own, c)  \
    BSI_I8_KSTEP_AT(0, here, acc, prev, qs);                \
    lds_barrier();                                          \
    BSI_I8_KSTEP_AT(1, (here) + C::kStage, acc, prev, qs);  \
    BSI_TILES_SCALES(own, c);                               \
    __builtin_amdgcn_sched_barrier(0);                      \
    BSI_I8_KSTEP_AT(2, (here) + C::kStage, acc, prev, qs);  \
    lds_barrier();                                          \
    BSI_I8_KSTEP_AT(3, next, acc, prev, qs);
#define BSI_I8_KSTEP_AT(KS, at, acc, prev, qs)                                                                              \
    i8_kstep<WM, WN, KS, kMode, false>(ka[(KS) & 1], qb[(KS) & 1], ka[((KS) + 1) & 1], qb[((KS) + 1) & 1],                  \
                                       lds + (at) + krow_off + pcol[((KS) + 1) & 1],                                        \
                                       lds + (at) + qrow_off + pcol[((KS) + 1) & 1], acc, prev, accf, qs, nullptr, int_off, \
                                       int_rows, down_shift, chunks, peak);
#define BSI_TILES_SCALES(dst, c)                                                               \
    {                                                                                          \
        _Pragma("unroll") for (int b = 0; b < WN; ++b) dst[b] =                                \
            *reinterpret_cast<const float*>(sread + ((c) & 3) * (C::kLoaders * 256) + b * 64); \
    }
    lds_barrier();  // stage 0 is there
#pragma unroll
    for (int t = 0; t < WM; ++t) ka[0][t] = *reinterpret_cast<const v4i*>(lds + krow_off + t * 16 * 128 + pcol[0]);
#pragma unroll
    for (int t = 0; t < WN; ++t) qb[0][t] = *reinterpret_cast<const v4i*>(lds + qrow_off + t * 16 * 128 + pcol[0]);
    __builtin_amdgcn_sched_barrier(0);
    int tile = 0;
#pragma nounroll
    for (unsigned id = blockIdx.x; id < tiles; id += gridDim.x, ++tile) {
        int c = 0;
        for (; c + 1 < chunks; c += 2) {
            BSI_TILES_CHUNK(even, odd, acc0, acc1, qsb, qsa, chunk0 + c);
            BSI_TILES_CHUNK(odd, even, acc1, acc0, qsa, qsb, chunk0 + c + 1);
        }
        // the chain step of the last chunk; the last k-step has read the next tile's first operands
        if (c < chunks) {
            BSI_TILES_CHUNK(even, odd, acc0, acc1, qsb, qsa, chunk0 + c);
            const int t = even;
            even = odd;
            odd = t;
#pragma unroll
            for (int a = 0; a < WM; ++a)
#pragma unroll
                for (int b = 0; b < WN; ++b)
#pragma unroll
                    for (int e = 0; e < 4; ++e) accf[a][b][e] = fmaf(static_cast<float>(acc0[a][b][e]), qsa[b], accf[a][b][e]);
        } else {
#pragma unroll
            for (int a = 0; a < WM; ++a)
#pragma unroll
                for (int b = 0; b < WN; ++b)
#pragma unroll
                    for (int e = 0; e < 4; ++e) accf[a][b][e] = fmaf(static_cast<float>(acc1[a][b][e]), qsb[b], accf[a][b][e]);
        }
        chunk0 += chunks;
        int bx, by;
        if (grid.height != 0) {
            i8_tile_of(grid, id, bx, by);
        } else {
            by = static_cast<int>(id / static_cast<unsigned>(grid.tiles_x));
            bx = static_cast<int>(id) - by * grid.tiles_x;
        }
        if constexpr (kLeft) by = left_tile(left, by);
        // from values the compiler cannot see through, so that no address of the stores is held in registers over the chunk loop
        int ln_late = ln, lg_late = lg;
        asm volatile("" : "+v"(ln_late), "+v"(lg_late));
        i8_store_tile<TM, WM, WN, kHalf>(accf, lds + 4 * C::kStage + I8TilesCfg<TM, TN>::kScaleBytes + (tile & 3) * C::kEpilogueBytes, down, scale_inv,
                                        bias != nullptr, out_dtype, out, R_total, static_cast<int64_t>(bx) * TM,
                                        static_cast<int64_t>(by) * TN, wr, wq, R, Q, ln_late, lg_late, out_stream != 0);
#pragma unroll
        for (int b = 0; b < WN; ++b) qsb[b] = 0.0f;  // the first chunk's chain step adds nothing
#pragma unroll
        for (int a = 0; a < WM; ++a)
#pragma unroll
            for (int b = 0; b < WN; ++b)
#pragma unroll
                for (int e = 0; e < 4; ++e) accf[a][b][e] = 0.0f;
    }
#undef BSI_TILES_CHUNK
#undef BSI_I8_KSTEP_AT
#undef BSI_TILES_SCALES
}

// ------------------------------------------------------------------ int8 image, 256 x 256 tiles of plain integer sums
//
// Large layers.  A chunk's scale is a power of two, and the integers of a row times its chunks' scales are multiples of the
// smallest of them: written in that unit, most are int8 still -- the chunks of a row differ by a factor of two, the int8 image
// has a bit to spare -- and the few that are not (outlier columns) keep their upper digit in a second image of which only the
// blocks of 64 elements are read that have one.  The dot is then ONE int32 sum over the row, and if the row's magnitudes
// times the largest key magnitude add up to no more than 2^24 units, every value the fp32 chain over the chunks takes is an
// integer of at most 24 bits: it never rounds, and the sum is its result, bit for bit.  i8_units_kernel writes the images, the
// masks of the blocks and the rows' units and checks that bound; a band of 256 queries with a row outside it, or with more
// than a quarter of its blocks in the second image, is left to the chain, in a launch behind this one that has those bands' tiles
// only and ends at once where there are none.  large_bands_kernel says so of each band ahead of the launch, and each workgroup
// works out the same two things from it: which bands are kept -- their tiles are numbered through, so that they fill the rounds of
// workgroups of every XCD -- and whether the chain had better take all, as a launch of one round is no shorter for the bands it leaves.
// us a layer, 0, 1, a quarter, half and all of the bands left, and tiles of 128 x 128: 4096 x 4096 x 16384 bf16 246, 264, 265, 282, 302,
// 284; 2048 x 8192 x 8192 f32 141, 164, 163, 164, 163, 149; 4096 x 3072 x 16384 f16 199, 217, 217, 228, 245, 226; 1024 x 4096 x 16384 bf16
// 76, 86, 86, 86, 86, 77.  (All tiles in the chain wherever one band was left: 1.8 times the time of none.  Tiles of the kept bands where
// they lie in the matrix: 4096 x 4096 x 16384, a quarter 302, half 356.)  What a layer loses of which nothing is kept is the images, 8,
// and two launches.
//
// Without the chain there are no second accumulators and no scales, a wave holds 128 x 64 outputs and a workgroup 256 x 256:
// half the bytes from the L2 and two thirds of the LDS reads a multiply-add, both of which the clock pays for.  Eight waves that load
// for themselves (eight loads a half-chunk among 64 MFMAs; two waves a SIMD leave room for no others); LDS is a ring of five
// slots of an operand's half-chunk, 256 rows x 128 bytes: K runs three stages ahead, Q two.
// us a layer with its build, tiles of 128 x 128 and now: 4096 x 4096 x 16384 bf16 283, 246 (this kernel 222); 2048 x 8192 x 8192 f32 152,
// 141; 4096 x 3072 x 16384 f16 227, 199; 1024 x 4096 x 16384 bf16 78, 76.  Of the launch's 483 k cycles the matrix pipes are busy in 280 k.
// A tile of 4096 (stamps): 4 to 5 us until its first stage is there and 4.2 for its stores, at 2.1 to 2.4 GHz with the pipes idle, 41 to 47
// of loop at 1.75 to 1.87, 2260 to 2410 cycles a stage and 2048 of them MFMA.  Tried beside it: touching
// lines of later stages ahead of their loads (260 -> 275, the loads are not what is waited for), the loads in one run behind the
// barrier (260 -> 267 -> 275 with their offsets worked out there too).
constexpr int kLargeSlot = kLargeTile * 128, kLargeSlots = 5, kLargeLds = kLargeSlots * kLargeSlot;
constexpr int kLargeMaskWords = 4, kLargeMaxChunks = 16 * kLargeMaskWords;  // 64-element blocks of a row, 64 a word
constexpr uint32_t kNowhere = 0x80000000u;  // past the end of every operand

// The images in units and what the dot needs to know of a row.  lo / hi: [Q][chunks * 256]; masks: [Q][words] of 64 blocks;
// units: [Q], the factor of the row's sums, negative where the row has to go through the chain.
// Four elements in units: their bytes in either image.  exponent: of their scale, 255 where all are zero; least: of the row's unit.
__device__ __forceinline__ void unit_bytes(uint32_t in, unsigned exponent, unsigned least, int Sa, uint32_t& low_bytes, uint32_t& high_bytes,
                                           unsigned& total, unsigned& odd) {
    int up = exponent == 255u ? 0 : static_cast<int>(exponent - least) - (8 - Sa);  // the image holds a << (8 - Sa)
    if (up <= 0) {  // nearly all: every element is in the lower image, the four of them shifted together
        const uint32_t sign = in >> 7 & 0x01010101u, keep = (0xFFu >> -up) * 0x01010101u;
        low_bytes = (in >> -up & keep) | sign * (0xFFu & ~(0xFFu >> -up));
        high_bytes = 0u;
        total = __builtin_amdgcn_sad_u8(low_bytes ^ 0x80808080u, 0x80808080u, total);  // |a| is the distance of a + 128 and 128
        return;
    }
    if (up > 8) {
        odd = 1u;
        up = 8;
    }
    low_bytes = high_bytes = 0u;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int a = (static_cast<int>(in << (24 - 8 * k)) >> 24) << up;
        const int low = static_cast<int>(static_cast<uint32_t>(a) << 24) >> 24;
        total += static_cast<unsigned>(a < 0 ? -a : a);
        low_bytes |= (static_cast<uint32_t>(a) & 255u) << (8 * k);
        high_bytes |= (static_cast<uint32_t>((a - low) >> 8) & 255u) << (8 * k);
    }
}
// The factor of a row's sums, from what its waves have found; leaves with all of them past a barrier.
template <int kWaves>
__device__ __forceinline__ void unit_of_row(unsigned (&shared)[3][kWaves], int lane, int wave, unsigned total, unsigned odd, unsigned least, int Sb,
                                            float* __restrict__ unit) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) total += __shfl_xor(total, o, BSI_WAVE);
    const bool any_odd = __ballot(odd != 0u) != 0ull;
    if (lane == 0) {
        shared[1][wave] = total;
        shared[2][wave] = any_odd ? 1u : 0u;
    }
    __syncthreads();
    if (wave == 0 && lane == 0) {
        unsigned long long sum = 0ull;
        unsigned bad = 0u;
        for (int w = 0; w < kWaves; ++w) {
            sum += shared[1][w];
            bad |= shared[2][w];
        }
        if (least == 255u) least = 127u;  // a row of zeros
        // the key image holds b << (8 - Sb), |b| <= 2^(Sb - 1)
        *unit = bad != 0u || (sum << (Sb - 1)) > (1ull << 24) ? -1.0f : __uint_as_float((least - static_cast<unsigned>(8 - Sb)) << 23);
    }
}
constexpr int kUnitsBlock = 256, kUnitsHeld = kLargeMaxChunks * 16 / kUnitsBlock;
__global__ __launch_bounds__(kUnitsBlock) void i8_units_kernel(const int8_t* __restrict__ A8, const float* __restrict__ qscale, int stride,
                                                               int chunks, int Sa, int Sb, uint4* __restrict__ lo, uint4* __restrict__ hi,
                                                               unsigned short* __restrict__ masks, float* __restrict__ units) {
    constexpr int kUnitsWaves = kUnitsBlock / 64;
    __shared__ unsigned shared[3][kUnitsWaves];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t row = blockIdx.x;
    const int pieces = chunks * 16, mask_pieces = (chunks * 4 + 63) / 64 * 4;  // of 16 bytes; of 16 mask bits
    const uint4* const src = reinterpret_cast<const uint4*>(A8) + row * pieces;
    const float* const scales = qscale + row * stride;
    uint4 v[kUnitsHeld];
    unsigned exponent[kUnitsHeld], least = 255u, odd = 0u;  // of the scales of pieces that are not all zero
#pragma unroll
    for (int j = 0; j < kUnitsHeld; ++j) {
        const int p = tid + j * kUnitsBlock;
        v[j] = make_uint4(0u, 0u, 0u, 0u);
        exponent[j] = 255u;
        if (p >= pieces) continue;
        v[j] = src[p];
        const unsigned bits = __float_as_uint(scales[stride == 1 ? 0 : p >> 4]);
        if ((v[j].x | v[j].y | v[j].z | v[j].w) == 0u) continue;
        if ((bits & 0x807FFFFFu) != 0u || bits < 0x20000000u || bits >= 0x60000000u) odd = 1u;  // no power of two, or a far one
        exponent[j] = bits >> 23 & 255u;
        least = exponent[j] < least ? exponent[j] : least;
    }
    least = ~wave_max_u32(~least);
    if (lane == 0) shared[0][wave] = least;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kUnitsWaves; ++w) least = shared[0][w] < least ? shared[0][w] : least;
    unsigned total = 0u;  // of the row's magnitudes, in units: at most 2^14 elements of 2^15
#pragma unroll
    for (int j = 0; j < kUnitsHeld; ++j) {
        const int p = tid + j * kUnitsBlock, at = wave + j * kUnitsWaves;
        if (at >= mask_pieces) break;  // the whole wave
        uint32_t l[4], h[4];
        const uint32_t in[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
#pragma unroll
        for (int i = 0; i < 4; ++i) unit_bytes(in[i], exponent[j], least, Sa, l[i], h[i], total, odd);
        // four neighbouring lanes hold a block of 64 elements
        const unsigned long long any = __ballot((h[0] | h[1] | h[2] | h[3]) != 0u);
        unsigned long long m = (any | any >> 1 | any >> 2 | any >> 3) & 0x1111111111111111ull;
        m = (m | m >> 3) & 0x0303030303030303ull;
        m = (m | m >> 6) & 0x000F000F000F000Full;
        m = (m | m >> 12) & 0x000000FF000000FFull;
        m = (m | m >> 24) & 0xFFFFull;
        if (lane == 0) masks[row * mask_pieces + at] = static_cast<unsigned short>(m);
        if (p < pieces) {
            lo[row * pieces + p] = make_uint4(l[0], l[1], l[2], l[3]);
            hi[row * pieces + p] = make_uint4(h[0], h[1], h[2], h[3]);
        }
    }
    unit_of_row<kUnitsWaves>(shared, lane, wave, total, odd, least, Sb, units + row);
}

// The same with the build: a workgroup quantises a row, a chunk a wave at a time, and has the row's unit before it stores the
// chunks.  For layers with chunk scales; writes what build_fixed_chunk_fast_kernel and then i8_units_kernel do, and does not read the
// image, which only the chain looks at, again.  us, those two and this: 4096 x 4096 bf16 26.9, 22.3 (84 MB, 3.8 TB/s; 23.8 with the
// shifts of unit_bytes an element at a time); a layer 4096 x 4096 x 16384 bf16 249, 245; 1024 x 4096 x 16384 70.3, 67.9; 2048 x 8192
// x 8192 f32 134.4, 132; 4096 x 3072 x 16384 f16 211, 205.
template <typename T, bool kVec, int kHeld>
__global__ __launch_bounds__(kUnitsBlock) void build_units_kernel(const T* __restrict__ x, int64_t d, int chunks, int Sa, int Sb, double dec_scale,
                                                                  float scale, int* __restrict__ shifts, float* __restrict__ scales,
                                                                  uint32_t* __restrict__ image, uint32_t* __restrict__ lo, uint32_t* __restrict__ hi,
                                                                  unsigned long long* __restrict__ masks, float* __restrict__ units) {
    constexpr int kUnitsWaves = kUnitsBlock / 64;
    __shared__ unsigned shared[3][kUnitsWaves];
    __shared__ unsigned blocks[kLargeMaxChunks];  // of a chunk, which of its four blocks are in the upper image
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const size_t row = blockIdx.x;
    const T* const src = x + row * static_cast<size_t>(d);
    const ChunkLane cl = chunk_lane(lane);
    const QuantRange range = quant_range(Sa);
    if (tid < kLargeMaxChunks) blocks[tid] = 0u;
    float v[kHeld][4];
#pragma unroll
    for (int j = 0; j < kHeld; ++j) load_chunk_quad<T, kVec>(src, d, wave + j * kUnitsWaves, cl, v[j]);  // past the row: zeros
    uint32_t held[kHeld];
    unsigned exponent[kHeld], least = 255u, odd = 0u, total = 0u;
#pragma unroll
    for (int j = 0; j < kHeld; ++j) {
        const int c = wave + j * kUnitsWaves;
        held[j] = 0u;
        exponent[j] = 255u;
        if (c >= chunks) continue;
        const unsigned mx = wave_max_u32(quad_max_bits(v[j]));
        int shift;
        uint32_t bytes;
        if (mx < kQuantWideBits) {
            shift = quant_shift(mx, scale, Sa);
            bytes = quantise_quad<T>(v[j], scale, shift, range);
        } else {
            shift = compute_shift(wave_max_u64(quad_max_wide(v[j], dec_scale)), 0.0, BSI_CHUNK_ELEMS, Sa, 0.0f);
            bytes = quantise_quad_wide(v[j], dec_scale, shift, Sa);
        }
        held[j] = chunk_image_dword(bytes, cl);
        image[(row * chunks + c) * 64 + lane] = held[j];
        if (lane == 0) {
            shifts[row * chunks + c] = shift;
            scales[row * chunks + c] = static_cast<float>(1ULL << shift);
        }
        if (__ballot(held[j] != 0u) != 0ull) exponent[j] = static_cast<unsigned>(127 + shift);
        least = exponent[j] < least ? exponent[j] : least;
    }
    if (lane == 0) shared[0][wave] = least;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kUnitsWaves; ++w) least = shared[0][w] < least ? shared[0][w] : least;
#pragma unroll
    for (int j = 0; j < kHeld; ++j) {
        const int c = wave + j * kUnitsWaves;
        if (c >= chunks) break;
        uint32_t l, h;
        unit_bytes(held[j], exponent[j], least, Sa, l, h, total, odd);
        const unsigned long long any = __ballot(h != 0u);
        if (lane == 0)
            blocks[c] = ((any & 0xFFFFull) != 0ull ? 1u : 0u) | ((any & 0xFFFF0000ull) != 0ull ? 2u : 0u) |
                        ((any & 0xFFFF00000000ull) != 0ull ? 4u : 0u) | (any >> 48 != 0ull ? 8u : 0u);
        lo[(row * chunks + c) * 64 + lane] = l;
        hi[(row * chunks + c) * 64 + lane] = h;
    }
    unit_of_row<kUnitsWaves>(shared, lane, wave, total, odd, least, Sb, units + row);
    const int words = (chunks * 4 + 63) / 64;
    if (tid < words) {
        unsigned long long m = 0ull;
#pragma unroll
        for (int i = 0; i < 16; ++i) m |= static_cast<unsigned long long>(blocks[tid * 16 + i]) << (4 * i);
        masks[row * words + tid] = m;
    }
}

// The stages of a tile: its blocks in the upper image, two of any place a stage, then the half-chunks of the lower one.
struct LargeStages {
    unsigned long long mask[kLargeMaskWords];
    int base, upper, half, halves;  // first block of mask[0]; stages left in the upper image; half-chunk to come; of the row
    __device__ __forceinline__ uint32_t block() {  // byte offset inside a row of the next block of the upper image
#pragma unroll
        for (int i = 0; i < kLargeMaskWords; ++i)
            if (mask[0] == 0ull) {
#pragma unroll
                for (int w = 0; w + 1 < kLargeMaskWords; ++w) mask[w] = mask[w + 1];
                mask[kLargeMaskWords - 1] = 0ull;
                base += 64;
            }
        if (mask[0] == 0ull) return kNowhere;
        const int bit = __builtin_ctzll(mask[0]);
        mask[0] &= mask[0] - 1ull;
        return static_cast<uint32_t>(base + bit) * 64u;
    }
    // the next stage: where its two 64-byte columns lie, and whether in the upper image
    __device__ __forceinline__ bool next(uint32_t& first, uint32_t& second) {
        if (upper > 0) {
            --upper;
            first = block();
            second = block();
            return true;
        }
        first = half < halves ? static_cast<uint32_t>(half) * 128u : kNowhere;
        second = first + 64u;
        ++half;
        return false;
    }
};

// The bands of kLargeTile queries, a workgroup each: which blocks are in the upper image for any of a band's rows, and how many stages
// they are, or kToChain.
constexpr unsigned kToChain = ~0u;
__global__ __launch_bounds__(kLargeTile) void large_bands_kernel(const unsigned long long* __restrict__ masks, const float* __restrict__ units, int chunks,
                                                                 int64_t Q, unsigned long long* __restrict__ bands, unsigned* __restrict__ uppers) {
    constexpr int kWaves = kLargeTile / 64;
    __shared__ unsigned long long ored[kWaves][kLargeMaskWords];
    __shared__ unsigned bad[kWaves];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, words = (chunks * 4 + 63) / 64;
    const int64_t q = static_cast<int64_t>(blockIdx.x) * kLargeTile + tid;
    const bool mine = q < Q;
    const bool odd = mine && units[q] < 0.0f;
    unsigned long long m[kLargeMaskWords];
#pragma unroll
    for (int w = 0; w < kLargeMaskWords; ++w) m[w] = mine && w < words ? masks[q * words + w] : 0ull;
#pragma unroll
    for (int w = 0; w < kLargeMaskWords; ++w)
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) m[w] |= __shfl_xor(m[w], o, BSI_WAVE);
    const bool any_odd = __ballot(odd) != 0ull;
    if (lane == 0) {
#pragma unroll
        for (int w = 0; w < kLargeMaskWords; ++w) ored[wave][w] = m[w];
        bad[wave] = any_odd ? 1u : 0u;
    }
    __syncthreads();
    if (tid != 0) return;
    unsigned chain = 0u;
    int blocks = 0;
    for (int w = 0; w < kLargeMaskWords; ++w) {
        unsigned long long all = 0ull;
        for (int i = 0; i < kWaves; ++i) all |= ored[i][w];
        bands[static_cast<size_t>(blockIdx.x) * kLargeMaskWords + w] = all;
        blocks += __builtin_popcountll(all);
    }
    for (int i = 0; i < kWaves; ++i) chain |= bad[i];
    uppers[blockIdx.x] = chain != 0u || blocks > chunks ? kToChain : static_cast<unsigned>(blocks + 1) / 2;  // at most a quarter of the 4 chunks blocks
}

// What decides between the sums for some bands and the chain for all, in us (i8_large_serves): a round of workgroups of the sums and a
// stage more in it, a round of the chain, the chain for all; tiles of either kernel beside one another.
struct LargeCost {
    float round, stage, chain, whole;
    int across, small;
};

template <bool kHalf>
__global__ __launch_bounds__(512, 2) void dot_mfma_i8_large_kernel(
    const int8_t* lo, const int8_t* hi, const unsigned long long* __restrict__ bands, const unsigned* __restrict__ uppers, LargeCost cost,
    const float* __restrict__ units, const int8_t* K8, const float* __restrict__ Bw, int Sb, int chunks, int64_t R, int64_t Q, float scale_inv,
    int64_t R_total, float* __restrict__ out, const float* __restrict__ bias, const unsigned char* __restrict__ warm, long long warm_lines,
    int out_stream, I8Grid grid, int out_dtype, unsigned* __restrict__ left) {
    // bands, uppers: of large_bands_kernel.  left: the list of the bands that the chain takes, for dot_mfma_i8_tiles_kernel behind this launch:
    // those that large_bands_kernel has turned down, or all, where the sums for the others would not pay.
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];  // kLargeLds
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave & 1, wq = wave >> 1, ln = lane & 15, lg = lane >> 4;
    const unsigned all_bands = static_cast<unsigned>(grid.tiles_y);
    unsigned count = 0u, more = 0u;
    for (unsigned t = 0; t < all_bands; t += 64) {
        const unsigned u = t + lane < all_bands ? uppers[t + lane] : 0u;
        count += __builtin_popcountll(__ballot(u == kToChain));
        more += u == kToChain ? 0u : u;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) more += __shfl_xor(more, o, BSI_WAVE);
    const unsigned kept = all_bands - count, rounds = (kept * static_cast<unsigned>(cost.across) + 255u) / 256u;
    const unsigned chained = (2u * count * static_cast<unsigned>(cost.small) + 255u) / 256u;
    const float sums = static_cast<float>(rounds) * (cost.round + cost.stage * static_cast<float>(more) / static_cast<float>(kept > 0u ? kept : 1u)) - 8.0f;
    const bool all = kept == 0u || sums + static_cast<float>(chained) * cost.chain > cost.whole;
    if (blockIdx.x == 0 && wave == 0) {
        unsigned at = 1u;
        for (unsigned t = 0; t < all_bands; t += 64) {
            const bool listed = t + lane < all_bands && (all || uppers[t + lane] == kToChain);
            const unsigned long long m = __ballot(listed);
            if (listed) left[at + __builtin_popcountll(m & ((1ull << lane) - 1ull))] = t + lane;
            at += __builtin_popcountll(m);
        }
        if (lane == 0) left[0] = at - 1u;
    }
    // the tiles of the bands that are kept, numbered through as if there were no others: an XCD's run of them is as long as another's
    if (all || blockIdx.x >= kept * static_cast<unsigned>(grid.tiles_x)) return;
    if (count != 0u) narrow_grid(grid, static_cast<int>(kept));
    int bx, by;
    i8_tile_of(grid, blockIdx.x, bx, by);
    if (count != 0u) {
        int before = by;
        for (unsigned t = 0; t < all_bands; t += 64) {
            const bool keep = t + lane < all_bands && uppers[t + lane] != kToChain;
            const unsigned long long m = __ballot(keep);
            const int here = __builtin_popcountll(m);
            if (before < here) {
                by = static_cast<int>(t) + __builtin_ctzll(__ballot(keep && __builtin_popcountll(m & ((1ull << lane) - 1ull)) == before));
                break;
            }
            before -= here;
        }
    }
    const int64_t r0 = static_cast<int64_t>(bx) * kLargeTile, q0 = static_cast<int64_t>(by) * kLargeTile;
    const uint32_t rowbytes = static_cast<uint32_t>(chunks) << 8;
    const bsi_rsrc rk = make_rsrc(K8 + static_cast<size_t>(r0) * rowbytes, static_cast<size_t>(R - r0) * rowbytes);
    const bsi_rsrc rlo = make_rsrc(lo + static_cast<size_t>(q0) * rowbytes, static_cast<size_t>(Q - q0) * rowbytes);
    const bsi_rsrc rhi = make_rsrc(hi + static_cast<size_t>(q0) * rowbytes, static_cast<size_t>(Q - q0) * rowbytes);

    LargeStages stages;
#pragma unroll
    for (int w = 0; w < kLargeMaskWords; ++w) stages.mask[w] = bands[static_cast<size_t>(by) * kLargeMaskWords + w];
    stages.base = stages.half = 0;
    stages.upper = static_cast<int>(uppers[by]);
    stages.halves = 2 * chunks;
    const int upper_stages = stages.upper;

    // loads: a wave moves rows 32 wave .. + 31 of an operand's stage, four loads of 8 rows x 128 bytes; lane = (row of the eight,
    // 16-byte column), columns swizzled as in dot_mfma_i8_kernel
    const uint32_t lr = static_cast<uint32_t>(lane) >> 3, lc = static_cast<uint32_t>(lane) & 7;
    uint32_t col[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) col[p] = lc ^ (static_cast<uint32_t>(p) * 4 + (lr >> 1));
    const uint32_t row0 = (static_cast<uint32_t>(wave) * 32 + lr) * rowbytes, rows8 = 8 * rowbytes;
    auto load = [&](bsi_rsrc r, int slot, const uint32_t (&off)[2], int i) {  // load i of four
        load16_to_lds(r, off[i & 1] + static_cast<uint32_t>(i) * rows8, 0, lds + slot * kLargeSlot + wave * 4096 + i * 1024);
    };
    auto issue = [&](bsi_rsrc r, int slot, const uint32_t (&off)[2]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) load(r, slot, off, i);
    };
    // the offsets of the next stage, the same for either operand; returns whether it is in the upper image
    auto advance = [&](uint32_t (&off)[2]) {
        uint32_t first, second;
        const bool in_upper = stages.next(first, second);
#pragma unroll
        for (int p = 0; p < 2; ++p) off[p] = row0 + (col[p] & 3) * 16 + (col[p] >= 4 ? second : first);
        return in_upper;
    };
    v4i acc[8][4];
#pragma unroll
    for (int a = 0; a < 8; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[a][b] = (v4i){0, 0, 0, 0};
    const int koff = (wr * 128 + ln) * 128, qoff = (wq * 64 + ln) * 128;
    int pcol[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) pcol[kk] = ((kk * 4 + lg) ^ (ln >> 1)) * 16;
    v4i ka[2][8], qb[2][4];
    // K0 Q0 K1 Q1 K2 into slots 0 .. 4; then, when stage s has been read, Q of stage s + 2 and K of stage s + 3
    uint32_t off[2], late[2];  // offsets of the stage K comes from next, and Q
    bool upper = advance(off), late_upper;
    issue(rk, 0, off);
    issue(upper ? rhi : rlo, 1, off);
    upper = advance(off);
    issue(rk, 2, off);
    issue(upper ? rhi : rlo, 3, off);
    upper = advance(off);
    issue(rk, 4, off);
    asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
    lds_barrier();
    int sk = 0;  // slot of K of the stage; Q in the next one
#pragma unroll
    for (int b = 0; b < 4; ++b) qb[0][b] = *reinterpret_cast<const v4i*>(lds + kLargeSlot + qoff + b * 2048 + pcol[0]);
#pragma unroll
    for (int a = 0; a < 8; ++a) ka[0][a] = *reinterpret_cast<const v4i*>(lds + koff + a * 2048 + pcol[0]);
    __builtin_amdgcn_sched_barrier(0);
#define BSI_LARGE_KSTEP(cur, nxt, kbase, qbase, BESIDE)                                                                \
    _Pragma("unroll") for (int a = 0; a < 8; ++a) {                                                                    \
        _Pragma("unroll") for (int b = 0; b < 4; ++b) {                                                                \
            acc[a][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ka[cur][a], qb[cur][b], acc[a][b], 0, 0, 0);             \
            const int t = a * 4 + b;                                                                                   \
            if (t < 24 && (t & 1) == 0) {                                                                              \
                const int r = t >> 1;                                                                                  \
                if (r < 4) qb[nxt][r] = *reinterpret_cast<const v4i*>(lds + (qbase) + r * 2048);                       \
                else ka[nxt][r - 4] = *reinterpret_cast<const v4i*>(lds + (kbase) + (r - 4) * 2048);                   \
            }                                                                                                          \
            BESIDE;                                                                                                    \
            __builtin_amdgcn_sched_barrier(0);                                                                         \
        }                                                                                                              \
    }
    // A stage.  Where the loads behind the barrier come from is worked out among the MFMAs of the first k-step (NEXT: `off` of K goes
    // on to stage s + 3, that of Q is what it was), and they are issued among those of the second: in a run of their own they
    // leave the matrix pipes idle, as all waves come to them at the same time.  The wait: stage s + 1 has landed (K of stage s + 2
    // may be in flight); behind the barrier all of stage s has been read.
#define BSI_LARGE_STAGE(NEXT, from)                                                                                                  \
    {                                                                                                                              \
        const int sq = sk + 1 >= kLargeSlots ? sk + 1 - kLargeSlots : sk + 1;                                                      \
        const int nk = sk + 2 >= kLargeSlots ? sk + 2 - kLargeSlots : sk + 2, nq = sk + 3 >= kLargeSlots ? sk + 3 - kLargeSlots : sk + 3; \
        BSI_LARGE_KSTEP(0, 1, sk * kLargeSlot + koff + pcol[1], sq * kLargeSlot + qoff + pcol[1], if (t == 24) {                   \
            late[0] = off[0];                                                                                                      \
            late[1] = off[1];                                                                                                      \
            NEXT;                                                                                                                  \
        });                                                                                                                        \
        asm volatile("s_waitcnt vmcnt(4)" ::: "memory");                                                                           \
        lds_barrier();                                                                                                             \
        BSI_LARGE_KSTEP(1, 0, nk * kLargeSlot + koff + pcol[0], nq * kLargeSlot + qoff + pcol[0], {                                \
            if (t >= 1 && t < 9 && (t & 1) == 1) load(from, sk, late, t >> 1);                                                     \
            if (t >= 9 && t < 25 && (t & 3) == 1) load(rk, sq, off, (t - 9) >> 2);                                                 \
        });                                                                                                                        \
        sk = nk;                                                                                                                   \
    }
    if (upper_stages > 0) {
#pragma nounroll
        for (int s = 0; s < upper_stages; ++s) BSI_LARGE_STAGE(late_upper = upper; upper = advance(off), late_upper ? rhi : rlo);
        // their sums move up by their eight bits
#pragma unroll
        for (int a = 0; a < 8; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[a][b][e] <<= 8;
    }
    // the lower image: `off` is that of half-chunk 2
    uint32_t step = 128u;
    int ahead = 3;  // the half-chunk that K goes on to; past the last one nothing is read
#pragma nounroll
    for (int s = 0; s < 2 * chunks; ++s) {
        step = ahead == 2 * chunks ? kNowhere : (ahead > 2 * chunks ? 0u : 128u);
        ++ahead;
        BSI_LARGE_STAGE(off[0] += step; off[1] += step, rlo);
    }
#undef BSI_LARGE_STAGE
#undef BSI_LARGE_KSTEP
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __syncthreads();  // the ring is free
    float* const epi = reinterpret_cast<float*>(lds);
    if (tid < kLargeTile) {
        const int64_t r = r0 + tid;
        epi[tid] = r < R ? Bw[r * Sb] : 0.0f;
        epi[kLargeTile + tid] = (bias != nullptr && r < R) ? bias[r] : 0.0f;
    }
    float unit[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        const int64_t q = q0 + wq * 64 + b * 16 + ln;
        unit[b] = q < Q ? units[q] : 0.0f;
    }
    __syncthreads();
#pragma unroll
    for (int a0 = 0; a0 < 8; a0 += 2) {  // two 16-key tiles at a time: piece wr * 4 + a0 / 2 of the 256 keys
        float v[2][4][4];
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int e = 0; e < 4; ++e) v[a][b][e] = static_cast<float>(acc[a0 + a][b][e]) * unit[b];  // exact
        i8_store_tile<kLargeTile, 2, 4, kHalf>(v, lds, 1.0f, scale_inv, bias != nullptr, out_dtype, out, R_total, r0, q0, wr * 4 + a0 / 2, wq, R, Q,
                                               ln, lg, out_stream != 0);
    }
    if (warm_lines > 0) i8_warm_lines<8>(lds, wave, lane, warm, warm_lines);
}

// ------------------------------------------------------------------ int8 image, one accumulator set per MFMA wave
//
// The same workgroup tile (128 keys x 128 queries), ring and epilogue as dot_mfma_i8_kernel<128, 128>, with MFMA waves
// that keep ONE int32 accumulator set instead of two.  Without a second set to park a finished chunk in, the chain
// step of chunk c (one cvt + one fma per output) runs on the accumulators in place, between a tile's last MFMA of
// chunk c (k-step 3) and its first of chunk c + 1 (k-step 0, which starts from zero and overwrites it): two
// elements behind each MFMA of k-step 3 from its third MFMA on, three behind each of the first MFMAs of the next
// k-step 0, always of tiles whose turn to be overwritten has not come.  The 32 registers this frees per wave let four
// MFMA waves of 64 keys x 64 queries (WN = 4 query tiles; one wave per SIMD, 256 registers each) do the work of eight
// of 64 x 32: an MFMA wave's operand reads are (64 + 64) x 64 bytes per 64 x 64 x 64 MACs instead of (64 + 32) x 64
// per 64 x 32 x 64, a third fewer LDS bytes per MAC.  (The same scheme on eight MFMA waves of 64 x 32 with eight
// loader waves needs 16 waves of at most 128 registers; it spills and is slower, so it is not built.)
template <int WN>
struct I8WDump {  // where a lane's accumulators go in the [Q, R, chunks] dump (parity checks): element (a, b, e) at
    int64_t base, qstep;  // base + b * qstep + (a * 16 + e) * chunks, for the query columns of qmask and the
    int rows[4];          // first rows[a] key rows of tile a
    unsigned qmask;
};
template <int WN, bool kInts>
__device__ __forceinline__ void i8w_chain(int first, int count, const v4i (&acc)[4][WN], float (&accf)[4][WN][4],
                                          const float (&qs)[WN], int* __restrict__ ints_at, const I8WDump<WN>& dump,
                                          int down_shift, int chunks) {
#pragma unroll
    for (int i = first; i < first + count; ++i) {
        if (i >= 16 * WN) break;
        const int tile = i >> 2, e = i & 3, a = tile / WN, b = tile % WN;
        accf[a][b][e] = fmaf(static_cast<float>(acc[a][b][e]), qs[b], accf[a][b][e]);
        if (kInts && ints_at != nullptr && ((dump.qmask >> b) & 1u) && e < dump.rows[a])
            ints_at[dump.base + b * dump.qstep + static_cast<int64_t>(a * 16 + e) * chunks] = acc[a][b][e] >> down_shift;
    }
}

// One k-step of such an MFMA wave: 4 WN MFMAs (tile t = WN a + b), the reads of the next k-step's 4 + WN operand
// tiles behind the first of them, and the chain elements that fall to this k-step (see above).  qs_cur / ints_cur:
// scales and accumulator dump of the chunk being computed (used by k-step 3); qs_prev / ints_prev: of the chunk
// before it (used by k-step 0).
template <int WN, int KS, bool kInts>
__device__ __forceinline__ void i8w_kstep(const v4i (&ka)[4], const v4i (&qb)[WN], v4i (&ka_n)[4], v4i (&qb_n)[WN],
                                          const unsigned char* __restrict__ krow_n,
                                          const unsigned char* __restrict__ qrow_n, v4i (&acc)[4][WN],
                                          float (&accf)[4][WN][4], const float (&qs_cur)[WN], const float (&qs_prev)[WN],
                                          int* __restrict__ ints_cur, int* __restrict__ ints_prev, const I8WDump<WN>& dump,
                                          int down_shift, int chunks) {
    constexpr int NT = 4 * WN;            // tiles of the wave
    constexpr int kLate = 2 * (NT - 2);   // chain elements k-step 3 takes care of; the rest fall to the next k-step 0
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int a = t / WN, b = t % WN;
        const v4i c0 = (KS == 0) ? (v4i){0, 0, 0, 0} : acc[a][b];
        acc[a][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ka[a], qb[b], c0, 0, 0, 0);
        // read number t of the next k-step, in the order its MFMAs first need them: ka[0], qb[0 ..], ka[1 ..]
        if (t == 0) ka_n[0] = *reinterpret_cast<const v4i*>(krow_n);
        else if (t <= WN) qb_n[t - 1] = *reinterpret_cast<const v4i*>(qrow_n + (t - 1) * 16 * 128);
        else if (t < 4 + WN) ka_n[t - WN] = *reinterpret_cast<const v4i*>(krow_n + (t - WN) * 16 * 128);
        if (KS == 0 && kLate + 3 * t < 4 * NT)  // three elements of the previous chunk, of tiles above t
            i8w_chain<WN, kInts>(kLate + 3 * t, 3, acc, accf, qs_prev, ints_prev, dump, down_shift, chunks);
        if (KS == 3 && t >= 2)  // two elements of this chunk, of tiles finished two MFMAs ago or earlier
            i8w_chain<WN, kInts>(2 * (t - 2), 2, acc, accf, qs_cur, ints_cur, dump, down_shift, chunks);
        __builtin_amdgcn_sched_barrier(0);
    }
}

template <int WN>
struct I8WCfg {
    static_assert(WN == 4, "four MFMA waves of 64 x 64");
    using Tile = I8Cfg<128, 128>;  // LDS layout and loader waves
    static constexpr int kWavesN = 128 / (16 * WN);      // MFMA waves along the queries (2 along the keys)
    static constexpr int kConsumers = 2 * kWavesN;
    static constexpr int kBlock = (kConsumers + Tile::kLoaders) * 64;
};

template <int WN, bool kInts>
__global__ __launch_bounds__((I8WCfg<WN>::kBlock)) void dot_mfma_i8w_kernel(
    const int8_t* __restrict__ A8, const float* __restrict__ qscale, int qscale_stride, const int8_t* __restrict__ K8,
    const float* __restrict__ Bw, int Sb, int chunks, int64_t R, int64_t Q, int down_shift, float scale_inv,
    int64_t R_total, float* __restrict__ out, int* __restrict__ chunk_ints, const float* __restrict__ bias,
    int key_tiled, const unsigned char* __restrict__ warm, long long warm_lines, int out_stream, int out_dtype) {
    constexpr int TM = 128, TN = 128;
    using W = I8WCfg<WN>;
    using C = typename W::Tile;
    constexpr int kNE = 16 * WN;          // chain elements per lane and chunk
    constexpr int kLate = 2 * (4 * WN - 2);
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];  // C::kLds

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t r0 = static_cast<int64_t>(blockIdx.x) * TM;
    const int64_t q0 = static_cast<int64_t>(blockIdx.y) * TN;
    const size_t rowbytes = static_cast<size_t>(chunks) * 256;
    const int halves = chunks * 2;
    unsigned char* const scale_lds = lds + 4 * C::kStage;

    if (wave >= W::kConsumers) {
        i8_loader_wave<C, false, false>(lds, wave - W::kConsumers, lane, A8, qscale, qscale_stride, K8, Bw, Sb, chunks, 0, halves, R, Q,
                                 r0, q0, rowbytes, bias, 1, 0, key_tiled, warm, warm_lines);
        return;
    }

    // ---- MFMA waves: wr = half of the keys, wq = group of 16 WN queries
    const int wr = wave & 1, wq = wave >> 1;
    const int ln = lane & 15, lg = lane >> 4;
    const int krow_off = (wr * 64 + ln) * 128;
    const int qrow_off = C::kOperandK + (wq * (16 * WN) + ln) * 128;
    int pcol[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) pcol[kk] = ((kk * 4 + lg) ^ (ln >> 1)) * 16;
    float accf[4][WN][4];
    v4i acc[4][WN];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < WN; ++b) {
            acc[a][b] = (v4i){0, 0, 0, 0};
#pragma unroll
            for (int e = 0; e < 4; ++e) accf[a][b][e] = 0.0f;
        }
    const float down = __uint_as_float(static_cast<uint32_t>(127 - down_shift) << 23);
    I8WDump<WN> dump;
    {
        const int64_t rl = r0 + wr * 64 + lg * 4, ql = q0 + wq * (16 * WN) + ln;  // the lane's first key row and query column
        dump.base = (ql * R + rl) * chunks;
        dump.qstep = 16 * R * chunks;
        dump.qmask = 0;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const int64_t left = R - (rl + a * 16);
            dump.rows[a] = static_cast<int>(left < 0 ? 0 : (left < 4 ? left : 4));
        }
#pragma unroll
        for (int b = 0; b < WN; ++b)
            if (kInts && ql + b * 16 < Q) dump.qmask |= 1u << b;
    }
    // chunk scales of the lane's query columns, from the loaders' ring: 64 queries per region, region g = queries 64 g ..
    constexpr int sh = 0;
    const int qfirst = wq * (16 * WN);
    const unsigned char* sread = scale_lds + (qfirst >> 6) * 1024 + (((qfirst & 63) + ln) << (2 + sh));
    float qsa[WN], qsb[WN];  // scales of even / odd chunks (all zero before the first chunk: its "previous" chain adds 0)
#pragma unroll
    for (int b = 0; b < WN; ++b) qsa[b] = qsb[b] = 0.0f;
#define BSI_I8W_SCALES(dst, c)                                                                         \
    {                                                                                                  \
        _Pragma("unroll") for (int b = 0; b < WN; ++b) dst[b] =                                        \
            *reinterpret_cast<const float*>(sread + ((c) >> sh & 3) * C::kScaleGroup + ((c) & ((1 << sh) - 1)) * 4 + (b * 64 << sh)); \
    }
    v4i ka[2][4], qb[2][WN];  // operand sets of even / odd k-steps
#define BSI_I8W_KSTEP(KS, nslot, qc, qp, ic, ip)                                                                    \
    i8w_kstep<WN, KS, kInts>(ka[(KS) & 1], qb[(KS) & 1], ka[((KS) + 1) & 1], qb[((KS) + 1) & 1],                    \
                             lds + (nslot) * C::kStage + krow_off + pcol[((KS) + 1) & 1],                           \
                             lds + (nslot) * C::kStage + qrow_off + pcol[((KS) + 1) & 1], acc, accf, qc, qp, ic, ip, \
                             dump, down_shift, chunks);
    // a chunk whose halves sit in ring slots s0, s0 + 1; nslot: slot of the next chunk's first half; qc / qp: this
    // chunk's and the previous chunk's scales.  This chunk's scales have landed with its second half, which the
    // first barrier announces.
#define BSI_I8W_CHUNK(s0, nslot, qc, qp, ic, ip, c)                                                                 \
    BSI_I8W_KSTEP(0, s0, qc, qp, ic, ip);                                                                           \
    lds_barrier();                                                                                                  \
    BSI_I8W_SCALES(qc, c);                                                                                          \
    BSI_I8W_KSTEP(1, (s0) + 1, qc, qp, ic, ip);                                                                     \
    BSI_I8W_KSTEP(2, (s0) + 1, qc, qp, ic, ip);                                                                     \
    lds_barrier();                                                                                                  \
    BSI_I8W_KSTEP(3, nslot, qc, qp, ic, ip);

    lds_barrier();  // stage 0 is there
#pragma unroll
    for (int t = 0; t < 4; ++t) ka[0][t] = *reinterpret_cast<const v4i*>(lds + krow_off + t * 16 * 128 + pcol[0]);
#pragma unroll
    for (int t = 0; t < WN; ++t) qb[0][t] = *reinterpret_cast<const v4i*>(lds + qrow_off + t * 16 * 128 + pcol[0]);
    __builtin_amdgcn_sched_barrier(0);
    int c = 0;
    for (; c + 1 < chunks; c += 2) {
        // even chunk c: ring slots 0 and 1, scales qsa; the chain elements of chunk c - 1 left for its k-step 0 use qsb
        BSI_I8W_CHUNK(0, 2, qsa, qsb, chunk_ints + c, (c > 0 ? chunk_ints + (c - 1) : nullptr), c);
        // odd chunk c + 1: ring slots 2 and 3, scales qsb
        BSI_I8W_CHUNK(2, 0, qsb, qsa, chunk_ints + c + 1, chunk_ints + c, c + 1);
    }
    bool last_even = false;
    if (c < chunks) {  // odd number of chunks: one more even chunk
        BSI_I8W_CHUNK(0, 2, qsa, qsb, chunk_ints + c, (c > 0 ? chunk_ints + (c - 1) : nullptr), c);
        last_even = true;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the last k-step read ahead into a stage nothing uses
#undef BSI_I8W_CHUNK
#undef BSI_I8W_KSTEP
#undef BSI_I8W_SCALES
    // the chain elements of the last chunk that its k-step 3 left
    if (last_even) i8w_chain<WN, kInts>(kLate, kNE - kLate, acc, accf, qsa, chunk_ints + (chunks - 1), dump, down_shift, chunks);
    else i8w_chain<WN, kInts>(kLate, kNE - kLate, acc, accf, qsb, chunk_ints + (chunks - 1), dump, down_shift, chunks);
    // key factors and biases from the copy the loader waves staged in LDS
    float bs[4][4], bi[4][4];
    {
        const float* epi = reinterpret_cast<const float*>(lds + 4 * C::kStage + C::kScaleBytes);
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const int rl = wr * 64 + a * 16 + lg * 4;
            const float4 w4 = *reinterpret_cast<const float4*>(epi + rl);
            const float4 b4 = *reinterpret_cast<const float4*>(epi + TM + rl);
            bs[a][0] = key_factor(w4.x), bs[a][1] = key_factor(w4.y), bs[a][2] = key_factor(w4.z), bs[a][3] = key_factor(w4.w);
            bi[a][0] = b4.x, bi[a][1] = b4.y, bi[a][2] = b4.z, bi[a][3] = b4.w;
        }
    }
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < WN; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float v = ((accf[a][b][e] * down) * bs[a][e]) * scale_inv;
                if (bias != nullptr && out_dtype == BSI_DTYPE_F32) v = v + bi[a][e];
                accf[a][b][e] = v;
            }
    if (out_dtype != BSI_DTYPE_F32) {
        i8_store_half<4, WN>(accf, bi, bias != nullptr, out_dtype, out, R_total, r0 + wr * 64, q0 + wq * (16 * WN), R, Q, ln, lg);
        return;
    }
    i8_store_lines<4, WN>(accf, out, R_total, r0 + wr * 64, q0 + wq * (16 * WN), R, Q, ln, lg, out_stream != 0);
}

// out[q, idx[r]] = float(sum_{i,j} I[i Q + q, j R + r] * 2^(7 (i + j) - preshift) * Aw[q, 0] * Bw[r, 0]) * scale_inv
// (+ bias[r]): the digit products of the int32 GEMM put back together, exactly, in float64.
__global__ void digits_combine_kernel(const int* __restrict__ I, int nq, int nk, int64_t Q, int64_t R, int preshift,
                                      const float* __restrict__ Aw, int Sa, const float* __restrict__ Bw, int Sb,
                                      const long long* __restrict__ key_indices, float scale_inv, int64_t R_total,
                                      const float* __restrict__ bias, float* __restrict__ out) {
    const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (idx >= Q * R) return;
    const int64_t q = idx / R, r = idx - q * R;
    const int64_t ld = static_cast<int64_t>(nk) * R;
    double acc = 0.0;
    for (int i = 0; i < nq; ++i)
        for (int j = 0; j < nk; ++j)
            acc += ldexp(static_cast<double>(I[(static_cast<int64_t>(i) * Q + q) * ld + static_cast<int64_t>(j) * R + r]),
                         7 * (i + j) - preshift);
    acc = acc * static_cast<double>(Aw[q * Sa]) * static_cast<double>(Bw[r * Sb]);
    const int64_t col = key_indices ? key_indices[r] : r;
    float v = static_cast<float>(acc) * scale_inv;
    if (bias != nullptr) v = v + bias[r];
    out[q * R_total + col] = v;
}

// Set by bsi_hip_dot_bias_warm around its launch: the region the int8-image kernel should touch for the next dot.
thread_local const void* g_warm_ptr = nullptr;
thread_local size_t g_warm_bytes = 0;
// How the int8-image kernels store their output.  The entry points of a linear layer (bsi_hip_dot_bias,
// bsi_hip_dot_bias_warm, bsi_hip_linear) set t_layer_output around their launch: the next kernel of the model reads
// that output, so it is stored plainly and stays in the caches.  The dot entry points proper stream it out with
// nontemporal stores: the dirty lines then do not wait in the L2s for the write-back at the kernel's end (1.2 us less
// for the 16 MiB of Q512 R8192).  Measured both ways: streamed layer outputs cost an OPT-1.3B-shaped prefill 2 %
// (4.89 -> 5.00 ms replayed), plain dot outputs cost the standalone dot 8 %.  BSI_OPT_OUTPUT_STORES overrides.
// A layer's outputs are streamed as well from 80 MiB of float32 on, in rows of 2048 elements and more: that is more than the L2s hold
// (32 MiB) whoever reads them next, and on their way through the caches they push out keys that other tiles still need.  us a layer, and
// with torch.relu of its output behind it, plain and streamed: 2048 x 4096 x 11008 148, 113 and 176, 175; 2300 x 4096 x 11008 136, 126 and
// 167, 167; 4096 x 4096 x 16384 279, 268 and 359, 351 -- fewer outputs, and what the layer gains the next kernel loses: 1600 x 4096 x 11008
// (70 MB) 117, 92 and 136, 140; 4096 x 4096 x 4096 (67 MB) 95.6, 87.5 and 111, 113; shorter rows, whose tiles wait for their stores: 4096 x
// 256 x 5376 24.6, 26.0; 4096 x 512 x 8192 40.0, 40.2; 3000 x 512 x 16384 51.8, 52.0.
// Half-precision outputs have plain stores only: no difference up to 134 MB.
thread_local int t_layer_output = 0;
thread_local const CoopBuild* t_coop = nullptr;
thread_local int t_out_dtype = BSI_DTYPE_F32;
std::atomic<int> g_output_stores{0};  // 0 = by entry point, 1 = always plain, 2 = always nontemporal
constexpr int64_t kStreamedOutputs = 20 << 20;  // float32 outputs of a layer
constexpr int kStreamedChunks = 8;
int stream_output(int64_t R_total, int64_t Q, int chunks) {
    const int forced = g_output_stores.load(std::memory_order_relaxed);
    if (forced != 0) return forced == 2 ? 1 : 0;
    return t_layer_output && (R_total * Q < kStreamedOutputs || chunks < kStreamedChunks) ? 0 : 1;
}

constexpr int kCus = 256;

static I8Grid i8_bands(int64_t tiles_x, int64_t tiles_y, int64_t band) {  // in bands of about `band` query tiles
    const int64_t bands = (tiles_y + band - 1) / band, height = (tiles_y + bands - 1) / bands;
    auto reciprocal = [](int64_t n) { return n == 1 ? 0u : static_cast<unsigned>((int64_t{1} << 32) / n + 1); };
    return I8Grid{static_cast<int>(tiles_x), static_cast<int>(tiles_y), static_cast<int>(height), reciprocal(tiles_x * height),
                  reciprocal(height), reciprocal(tiles_y - (tiles_y - 1) / height * height)};
}

static I8Grid i8_grid(int64_t tiles_x, int64_t tiles_y, dim3* grid) {
    const I8Grid g = i8_bands(tiles_x, tiles_y, 8);  // 4 and 16 take the same time within 2 %
    // the reciprocals give exact quotients while dividend times divisor stays below 2^32
    if (tiles_x % 8 == 0 || tiles_x * tiles_y >= (int64_t{1} << 28) || tiles_x * tiles_y * tiles_x * g.height >= (int64_t{1} << 32)) {
        *grid = dim3(static_cast<unsigned>(tiles_x), static_cast<unsigned>(tiles_y));
        return I8Grid{static_cast<int>(tiles_x), static_cast<int>(tiles_y), 0, 0u, 0u, 0u};
    }
    *grid = dim3(static_cast<unsigned>(tiles_x * tiles_y));
    return g;
}

// The last round of a grid of 128 x 128 tiles, where it would leave half of the CUs idle: its tiles as quarters or halves, a CU each, in a
// launch of their own, which costs some 4 us and takes a round of 0.35 or 0.63.  Tiles of that launch, or 0.  us a layer in one launch and in
// two: up to 64 tiles, 4096 wide 281 x 12483 keys bf16 38.6, 34.5; 600 x 8192 bf16 35.8, 34.3; 1100 x 4096 f32 38.6, 37.3; 8192 wide 1100 x 4096 f32
// 69.8, 62.3; 600 x 8192 bf16 64.0, 58.5 -- 2048 wide 600 x 8192 f32 23.9, 24.8; up to 128 tiles, 8192 wide 768 x 8192 f32 82, 77; 3594 x 1536 bf16 84,
// 79 -- 4096 wide 768 x 8192 f32 39.9, 41.7; 777 x 11008 bf16 53.9, 53.6.
static int64_t i8_rest(int64_t tiles, int chunks) {
    const int64_t rest = tiles % kCus;
    if (tiles >= (1 << 22) || rest > kCus / 2) return 0;
    return chunks >= (rest <= kCus / 4 ? 12 : 24) ? rest : 0;
}
template <int TM, int TN, bool kFour, bool kHalf>
static void launch_mfma_i8_rest(int64_t first, int64_t rest, const I8Grid& g, const int8_t* A8, const float* qscale, int stride, const int8_t* K8,
                                const float* Bw, int Sb, int chunks, int64_t R, int64_t Q, int down_shift, float scale_inv, int64_t R_total,
                                float* out, const float* bias, hipStream_t st, int key_tiled) {
    using C = I8Cfg<TM, TN>;
    static LdsOptIn once;
    lds_opt_in(once, reinterpret_cast<const void*>(&dot_mfma_i8_kernel<TM, TN, kI8Chain, false, kParts, kFour, kHalf>), C::kLds);
    launch((dot_mfma_i8_kernel<TM, TN, kI8Chain, false, kParts, kFour, kHalf>), dim3(static_cast<unsigned>(rest * (128 / TM) * (128 / TN))), dim3(C::kBlock), C::kLds, st, A8,
           qscale, stride, K8, Bw, Sb, chunks, R, Q, down_shift, scale_inv, R_total, out, static_cast<int32_t*>(nullptr), bias, 0, 0LL,
           static_cast<const long long*>(nullptr), key_tiled, static_cast<const unsigned char*>(g_warm_ptr), static_cast<long long>(g_warm_bytes / 128),
           stream_output(R_total, Q, chunks), static_cast<float*>(nullptr), static_cast<unsigned*>(nullptr), 0.0f,
           static_cast<int>(rest | first << 8), g, t_out_dtype, CoopBuild{});
}

template <int TM, int TN, int kMode, bool kFour, bool kHalf>
static void launch_mfma_i8_tm(const int8_t* A8, const float* qscale, int stride, const int8_t* K8, const float* Bw,
                              int Sb, int chunks, int64_t R, int64_t Q, int down_shift, float scale_inv,
                              int64_t R_total, float* out, int32_t* chunk_ints, const float* bias, hipStream_t st,
                              int ndig, long long dig_stride, const long long* key_indices, int key_tiled) {
    using C = I8Cfg<TM, TN>;
    dim3 grid;
    const I8Grid g = i8_grid((R + TM - 1) / TM, (Q + TN - 1) / TN, &grid);
    const int64_t tiles = static_cast<int64_t>(g.tiles_x) * g.tiles_y;
    // more than one round of the large tiles, which fill a CU's LDS
    if constexpr (kMode == kI8Chain && TM == 128)
        if (t_coop == nullptr && tiles > kCus && tiles * chunks < (int64_t{1} << 29)) {
            static LdsOptIn once;
            lds_opt_in(once, reinterpret_cast<const void*>(&dot_mfma_i8_tiles_kernel<TM, TN, kHalf, false>), I8TilesCfg<TM, TN>::kLdsTiles);
            const int64_t rest = TN == 128 ? i8_rest(tiles, chunks) : 0;
            launch((dot_mfma_i8_tiles_kernel<TM, TN, kHalf, false>), dim3(kCus), dim3(C::kBlock), I8TilesCfg<TM, TN>::kLdsTiles, st, A8, qscale, stride,
                   K8, Bw, Sb, chunks, R, Q, down_shift, scale_inv, R_total, out, bias, key_tiled, static_cast<const unsigned char*>(g_warm_ptr),
                   rest != 0 ? 0LL : static_cast<long long>(g_warm_bytes / 128), stream_output(R_total, Q, chunks), g, static_cast<unsigned>(tiles - rest),
                   t_out_dtype, 0);
            if constexpr (TN == 128) {
                if (rest != 0)
                    (rest <= kCus / 4 ? &launch_mfma_i8_rest<64, 64, kFour, kHalf> : &launch_mfma_i8_rest<128, 64, kFour, kHalf>)(
                        tiles - rest, rest, g, A8, qscale, stride, K8, Bw, Sb, chunks, R, Q, down_shift, scale_inv, R_total, out, bias, st, key_tiled);
            }
            return;
        }
    if constexpr (kMode == kI8Chain)
        if (t_coop != nullptr) {
            CoopBuild coop = *t_coop;
            const unsigned all = coop_groups(grid.x * grid.y, R, coop, C::kBlock / 64);
            if (g.height != 0) grid.x = all;
            else grid.y = (all + grid.x - 1) / grid.x;
            coop.shares = coop_shares(all, coop.by_row ? coop.rows : coop.rows * coop.chunks, coop.shares);
            const auto go = [&](auto build) {
                constexpr int kBuild = decltype(build)::value;
                static LdsOptIn once;
                lds_opt_in(once, reinterpret_cast<const void*>(&dot_mfma_i8_kernel<TM, TN, kI8Chain, false, kBuild, false, kHalf>), C::kLds);
                launch((dot_mfma_i8_kernel<TM, TN, kI8Chain, false, kBuild, false, kHalf>), grid, dim3(C::kBlock), C::kLds, st, A8, qscale, stride, K8, Bw,
                       Sb, chunks, R, Q, down_shift, scale_inv, R_total, out, chunk_ints, bias, ndig, dig_stride, key_indices, key_tiled,
                       static_cast<const unsigned char*>(g_warm_ptr), static_cast<long long>(g_warm_bytes / 128), stream_output(R_total, Q, chunks),
                       static_cast<float*>(nullptr), static_cast<unsigned*>(nullptr), 0.0f, 0, g, t_out_dtype, coop);
            };
            if (coop.row_per_wave) go(std::integral_constant<int, 2>{});
            else go(std::integral_constant<int, 1>{});
            return;
        }
    static LdsOptIn once0;
    lds_opt_in(once0, reinterpret_cast<const void*>(&dot_mfma_i8_kernel<TM, TN, kMode, false, 0, kFour, kHalf>), C::kLds);
    launch((dot_mfma_i8_kernel<TM, TN, kMode, false, 0, kFour, kHalf>), grid, dim3(C::kBlock), C::kLds, st, A8, qscale, stride, K8,
                       Bw, Sb, chunks, R, Q, down_shift, scale_inv, R_total, out, chunk_ints, bias, ndig, dig_stride,
                       key_indices, key_tiled, static_cast<const unsigned char*>(g_warm_ptr),
                       static_cast<long long>(g_warm_bytes / 128), stream_output(R_total, Q, chunks), static_cast<float*>(nullptr),
                       static_cast<unsigned*>(nullptr), 0.0f, 0, g, t_out_dtype, CoopBuild{});
}

// The D-split launch of the chain mode: `segments` workgroups per output tile, each over its own run of chunks (see
// the head of dot_mfma_i8_kernel).  scratch: the calling thread's attached split scratch (counters, then partial sums).
template <int TM, int TN, bool kHalf>
static void launch_mfma_i8_split(int segments, unsigned char* scratch, const int8_t* A8, const float* qscale, int stride,
                                 const int8_t* K8, const float* Bw, int Sb, int chunks, int64_t R, int64_t Q, int down_shift,
                                 float scale_inv, int64_t R_total, float* out, const float* bias, hipStream_t st,
                                 int key_tiled) {
    using C = I8Cfg<TM, TN>;
    const int tiles_x = static_cast<int>((R + TM - 1) / TM), tiles_y = static_cast<int>((Q + TN - 1) / TN);
    const dim3 grid(static_cast<unsigned>(tiles_x * tiles_y * segments));
    const int split_shape = tiles_x | (tiles_y << 10) | (segments << 20);
    // every segment's chain values stay at or below 2^(24 + down_shift) / segments (rounded down to a power of two)
    int log2_segments = 0;
    while ((1 << log2_segments) < segments) ++log2_segments;
    const float limit = __builtin_ldexpf(1.0f, 24 + down_shift - log2_segments);
    static LdsOptIn once0;
    lds_opt_in(once0, reinterpret_cast<const void*>(&dot_mfma_i8_kernel<TM, TN, kI8Chain, true, 0, false, kHalf>), C::kLdsSplit);
    launch((dot_mfma_i8_kernel<TM, TN, kI8Chain, true, 0, false, kHalf>), grid, dim3(C::kBlock), C::kLdsSplit, st, A8, qscale,
                       stride, K8, Bw, Sb, chunks, R, Q, down_shift, scale_inv, R_total, out, static_cast<int*>(nullptr), bias,
                       1, 0LL, static_cast<const long long*>(nullptr), key_tiled,
                       static_cast<const unsigned char*>(g_warm_ptr), static_cast<long long>(g_warm_bytes / 128),
                       stream_output(R_total, Q, chunks), reinterpret_cast<float*>(scratch + kSplitCounterBytes),
                       reinterpret_cast<unsigned*>(scratch), limit, split_shape, I8Grid{}, t_out_dtype, CoopBuild{});
}

// Sum mode (ndig >= 1 digit images of the queries; int32 sums into chunk_ints when given, else the float epilogue)
// or, with ndig == 0, the chain with or without stored integers.
template <int TM, int TN>
static void launch_mfma_i8_t(int ndig, long long dig_stride, const long long* key_indices, int key_tiled, const int8_t* A8,
                             const float* qscale, int stride, const int8_t* K8, const float* Bw, int Sb, int chunks,
                             int64_t R, int64_t Q, int down_shift, float scale_inv, int64_t R_total, float* out,
                             int32_t* chunk_ints, const float* bias, hipStream_t st) {
    if (ndig > 0)
        launch_mfma_i8_tm<TM, TN, kI8Sum, false, false>(A8, qscale, stride, K8, Bw, Sb, chunks, R, Q, down_shift, scale_inv, R_total,
                                          out, chunk_ints, bias, st, ndig, dig_stride, key_indices, key_tiled);
    else if (chunk_ints)
        launch_mfma_i8_tm<TM, TN, kI8Ints, false, false>(A8, qscale, stride, K8, Bw, Sb, chunks, R, Q, down_shift, scale_inv, R_total,
                                           out, chunk_ints, bias, st, 1, 0, nullptr, key_tiled);
    else {
        const bool half = t_out_dtype != BSI_DTYPE_F32, four = i8_four_scales(stride);
#define BSI_I8_CHAIN(four_, half_) \
    launch_mfma_i8_tm<TM, TN, kI8Chain, four_, half_>(A8, qscale, stride, K8, Bw, Sb, chunks, R, Q, down_shift, scale_inv, R_total, out, \
                                                      chunk_ints, bias, st, 1, 0, nullptr, key_tiled)
        if (four) half ? BSI_I8_CHAIN(true, true) : BSI_I8_CHAIN(true, false);
        else half ? BSI_I8_CHAIN(false, true) : BSI_I8_CHAIN(false, false);
#undef BSI_I8_CHAIN
    }
}

// The 128 x 128 tile on four MFMA waves of 64 x 64 with one accumulator set, and four loader waves (tile 1284; chain
// modes only).
template <int WN>
static void launch_mfma_i8w(const int8_t* A8, const float* qscale, int stride, const int8_t* K8, const float* Bw, int Sb,
                            int chunks, int64_t R, int64_t Q, int down_shift, float scale_inv, int64_t R_total, float* out,
                            int32_t* chunk_ints, const float* bias, hipStream_t st, int key_tiled) {
    using W = I8WCfg<WN>;
    using C = typename W::Tile;
    const dim3 grid(static_cast<unsigned>((R + 127) / 128), static_cast<unsigned>((Q + 127) / 128));
    static LdsOptIn once0, once1;
    lds_opt_in(once0, reinterpret_cast<const void*>(&dot_mfma_i8w_kernel<WN, false>), C::kLds);
    lds_opt_in(once1, reinterpret_cast<const void*>(&dot_mfma_i8w_kernel<WN, true>), C::kLds);
    const unsigned char* warm = static_cast<const unsigned char*>(g_warm_ptr);
    const long long warm_lines = static_cast<long long>(g_warm_bytes / 128);
    if (chunk_ints)
        launch((dot_mfma_i8w_kernel<WN, true>), grid, dim3(W::kBlock), C::kLds, st, A8, qscale, stride, K8, Bw, Sb,
                           chunks, R, Q, down_shift, scale_inv, R_total, out, chunk_ints, bias, key_tiled, warm, warm_lines,
                           stream_output(R_total, Q, chunks), t_out_dtype);
    else
        launch((dot_mfma_i8w_kernel<WN, false>), grid, dim3(W::kBlock), C::kLds, st, A8, qscale, stride, K8, Bw, Sb,
                           chunks, R, Q, down_shift, scale_inv, R_total, out, chunk_ints, bias, key_tiled, warm, warm_lines,
                           stream_output(R_total, Q, chunks), t_out_dtype);
}

// The large layers' launches: the images in units, the bands, the integer sums, and the chain for what they leave.  The rule, in us: a round of
// 256 workgroups takes 1 a chunk and 1 with tiles of 128 x 128; with tiles of 256 x 256 2.95 a chunk and 2, and 8 more for each round
// but the last (all CUs store 32 MiB at the same time, with nothing else of theirs resident); the images are written at 0.75 a
// million elements; the launch that ends at once and the gaps are 14.  Measured, 128 x 128 and 256 x 256, bf16: taken 1024 x 4096 x
// 16384 73.6, 69.3; 4096 x 3072 x 16384 225, 207; 2048 x 8192 x 8192 150, 128.5; 1024 x 8192 x 16384 165, 123; not taken 4096 x 1024 x
// 16384 92, 99; 4096 x 2048 x 16384 155, 160; 4096 x 2048 x 8192 78, 85; 2048 x 4096 x 8192 74, 75 (f32 78, 81);
// 4096 x 4096 x 4096 78, 80; 3000 x 4096 x 11008 160, 172; and, at its edge, 2048 x 2048 x 16384 81, 77.  Float32 outputs that are streamed
// (stream_output), taken: 4096 x 4096 x 16384 313, 267; 4096 x 3072 x 16384 246, 224; 4096 x 4096 x 8192 156, 148; not taken: 4096 x 2048 x 16384
// 165, 168; 2048 x 2048 x 16384 88, 93; 2048 x 4096 x 11008 114, 128; 3000 x 4096 x 11008 166, 183; 4096 x 4096 x 6144 122, 142, and, where it would
// gain, 1536 x 8192 x 16384 238, 214; 2500 x 6144 x 8448 180, 173.
// A last round that runs as parts (i8_rest) is charged whole: charged as the parts take by themselves, layers would go to 128 x 128 that
// lose there.  128 x 128 with parts, and 256 x 256: bf16 2555 x 6144 x 5120 98.8, 96.1; 3276 x 8192 x 4096 142, 125; 3510 x 8192 x 3584 139, 127;
// 1287 x 5120 x 9472 85.2, 78.8; 3113 x 4096 x 9216 133, 128; f32 2555 x 6144 x 5120 114, 105; 3510 x 8192 x 3584 165, 140.
// Beyond 1 GiB of image the layer keeps to the workspace it had without units, which would be two more.
constexpr int64_t kLargeMaxItems = 1 << 22;  // (row, chunk) items
static size_t large_aligned(size_t v) { return (v + 255) / 256 * 256; }
size_t i8_large_workspace_bytes(int64_t Q, int chunks) {
    if (Q < kLargeMinQ || chunks > kLargeMaxChunks || Q > kLargeMaxItems / chunks) return 0;
    const size_t image = large_aligned(static_cast<size_t>(Q) * chunks * 256), words = static_cast<size_t>((chunks * 4 + 63) / 64);
    const size_t bands = static_cast<size_t>((Q + kLargeTile - 1) / kLargeTile);
    return 2 * image + large_aligned(static_cast<size_t>(Q) * words * 8) + large_aligned(static_cast<size_t>(Q) * 4) +
           large_aligned(bands * kLargeMaskWords * 8) + large_aligned(bands * 4) + large_aligned((bands + 1) * 4);
}

bool i8_large_serves(int64_t Q, int64_t R, int chunks) {
    const int forced = g_i8_tile.load(std::memory_order_relaxed);
    if (Q < kLargeMinQ || chunks > kLargeMaxChunks || Q > kLargeMaxItems / chunks || (forced != 0 && forced != kLargeTile)) return false;
    const int64_t small = ((R + 127) / 128) * ((Q + 127) / 128), large = ((R + kLargeTile - 1) / kLargeTile) * ((Q + kLargeTile - 1) / kLargeTile);
    // the tile kernels' own limits: ring positions and exact quotients in 32 bits
    if (small * chunks >= (int64_t{1} << 29) || large * ((R + kLargeTile - 1) / kLargeTile) >= (int64_t{1} << 29)) return false;
    if (forced == kLargeTile) return true;
    if (small <= kCus) return false;
    const double us_small = static_cast<double>((small + kCus - 1) / kCus) * (chunks + 1.0);
    const double us_large = static_cast<double>((large + kCus - 1) / kCus) * (2.95 * chunks + 10.0) + 6.0 + 7.5e-7 * static_cast<double>(Q) * chunks * 256;
    return us_large < us_small;
}

// The same figures for the sums of some bands beside the chain for the others; where the tile is asked for, the chain takes no more than it has to.
static LargeCost large_cost(int64_t Q, int64_t R, int chunks) {
    const int64_t small_x = (R + 127) / 128, small_y = (Q + 127) / 128;
    const float chain = static_cast<float>(chunks + 1);
    const bool forced = g_i8_tile.load(std::memory_order_relaxed) == kLargeTile;
    return LargeCost{2.95f * chunks + 10.0f, 1.475f, chain, forced ? INFINITY : chain * static_cast<float>((small_x * small_y + kCus - 1) / kCus),
                     static_cast<int>((R + kLargeTile - 1) / kLargeTile), static_cast<int>(small_x)};
}

struct LargeWorkspace {
    unsigned char *lo, *hi, *masks;
    float* units;
    unsigned char* bands;
    unsigned *uppers, *left;
};
static LargeWorkspace large_workspace(void* workspace, int64_t Q, int chunks) {
    const size_t image = large_aligned(static_cast<size_t>(Q) * chunks * 256), words = static_cast<size_t>((chunks * 4 + 63) / 64);
    LargeWorkspace w;
    w.lo = static_cast<unsigned char*>(workspace);
    w.hi = w.lo + image;
    w.masks = w.hi + image;
    w.units = reinterpret_cast<float*>(w.masks + large_aligned(static_cast<size_t>(Q) * words * 8));
    const size_t bands = static_cast<size_t>((Q + kLargeTile - 1) / kLargeTile);
    w.bands = reinterpret_cast<unsigned char*>(w.units) + large_aligned(static_cast<size_t>(Q) * 4);
    w.uppers = reinterpret_cast<unsigned*>(w.bands + large_aligned(bands * kLargeMaskWords * 8));
    w.left = reinterpret_cast<unsigned*>(w.bands + large_aligned(bands * kLargeMaskWords * 8) + large_aligned(bands * 4));
    return w;
}

template <typename T, bool kVec>
static void launch_build_units_t(const LargeWorkspace& w, const void* x, int64_t Q, int64_t d, int Sa, int Sb, double dec_scale, int32_t* shifts, float* scales,
                                 int8_t* ints8, int chunks, hipStream_t st) {
#define BSI_BUILD_UNITS(HELD)                                                                                                                       \
    launch((build_units_kernel<T, kVec, HELD>), dim3(static_cast<unsigned>(Q)), dim3(kUnitsBlock), 0, st, static_cast<const T*>(x), d, chunks, Sa, Sb, \
           dec_scale, static_cast<float>(dec_scale), shifts, scales, reinterpret_cast<uint32_t*>(ints8), reinterpret_cast<uint32_t*>(w.lo),          \
           reinterpret_cast<uint32_t*>(w.hi), reinterpret_cast<unsigned long long*>(w.masks), w.units)
    if (chunks <= 16) BSI_BUILD_UNITS(4);
    else if (chunks <= 32) BSI_BUILD_UNITS(8);
    else BSI_BUILD_UNITS(16);
#undef BSI_BUILD_UNITS
}
void launch_build_units(void* workspace, const void* x, int dtype, int64_t Q, int64_t d, int Sa, int Sb, double dec_scale, int32_t* shifts, float* scales,
                        int8_t* ints8, int chunks, hipStream_t st) {
    const LargeWorkspace w = large_workspace(workspace, Q, chunks);
    const bool vec = d % 4 == 0 && reinterpret_cast<uintptr_t>(x) % (dtype == BSI_DTYPE_F32 ? 16 : 8) == 0;
    const auto go = [&](auto zero) {
        using T = decltype(zero);
        (vec ? &launch_build_units_t<T, true> : &launch_build_units_t<T, false>)(w, x, Q, d, Sa, Sb, dec_scale, shifts, scales, ints8, chunks, st);
    };
    if (dtype == BSI_DTYPE_F32) go(float{});
    else if (dtype == BSI_DTYPE_F16) go(__half{});
    else go(__hip_bfloat16{});
}

template <bool kHalf>
static void launch_i8_large_t(const LargeWorkspace& w, bool units_there, const int8_t* A8, const float* qscale, int stride, const int8_t* K8,
                              const float* Bw, int Sa, int Sb, int chunks, int64_t R, int64_t Q, float scale_inv, int64_t R_total, float* out,
                              const float* bias, hipStream_t st) {
    if (!units_there)
        launch(i8_units_kernel, dim3(static_cast<unsigned>(Q)), dim3(kUnitsBlock), 0, st, A8, qscale, stride, chunks, Sa, Sb,
               reinterpret_cast<uint4*>(w.lo), reinterpret_cast<uint4*>(w.hi), reinterpret_cast<unsigned short*>(w.masks), w.units);
    const I8Grid g = i8_bands((R + kLargeTile - 1) / kLargeTile, (Q + kLargeTile - 1) / kLargeTile, 2);
    launch(large_bands_kernel, dim3(static_cast<unsigned>(g.tiles_y)), dim3(kLargeTile), 0, st, reinterpret_cast<const unsigned long long*>(w.masks), w.units,
           chunks, Q, reinterpret_cast<unsigned long long*>(w.bands), w.uppers);
    static LdsOptIn once, once_left;
    lds_opt_in(once, reinterpret_cast<const void*>(&dot_mfma_i8_large_kernel<kHalf>), kLargeLds);
    const unsigned char* const warm = static_cast<const unsigned char*>(g_warm_ptr);
    const long long warm_lines = static_cast<long long>(g_warm_bytes / 128);
    launch((dot_mfma_i8_large_kernel<kHalf>), dim3(static_cast<unsigned>(g.tiles_x) * static_cast<unsigned>(g.tiles_y)), dim3(512), kLargeLds, st,
           reinterpret_cast<const int8_t*>(w.lo), reinterpret_cast<const int8_t*>(w.hi), reinterpret_cast<const unsigned long long*>(w.bands),
           static_cast<const unsigned*>(w.uppers), large_cost(Q, R, chunks), w.units, K8, Bw, Sb, chunks, R, Q, scale_inv, R_total, out, bias, warm,
           warm_lines, stream_output(R_total, Q, chunks), g, t_out_dtype, w.left);
    dim3 grid;
    const I8Grid tiles = i8_grid((R + 127) / 128, (Q + 127) / 128, &grid);
    using T = I8TilesCfg<128, 128>;
    lds_opt_in(once_left, reinterpret_cast<const void*>(&dot_mfma_i8_tiles_kernel<128, 128, kHalf, true>), T::kLdsTiles);
    const int64_t left_tiles = static_cast<int64_t>(tiles.tiles_x) * tiles.tiles_y;  // of all bands; a workgroup without a tile ends before its first load
    launch((dot_mfma_i8_tiles_kernel<128, 128, kHalf, true>), dim3(static_cast<unsigned>(left_tiles < kCus ? left_tiles : kCus)), dim3(T::kBlock), T::kLdsTiles, st, A8, qscale, stride, K8, Bw, Sb, chunks,
           R, Q, 16 - Sa - Sb, scale_inv, R_total, out, bias, 0, warm, warm_lines, stream_output(R_total, Q, chunks), tiles,
           static_cast<unsigned>(left_tiles), t_out_dtype, w.left);
}
void launch_i8_large(void* workspace, bool units_there, const int8_t* A8, const float* qscale, int stride, const int8_t* K8, const float* Bw, int Sa, int Sb,
                     int chunks, int64_t R, int64_t Q, float scale_inv, int64_t R_total, float* out, const float* bias, hipStream_t st) {
    (t_out_dtype != BSI_DTYPE_F32 ? &launch_i8_large_t<true> : &launch_i8_large_t<false>)(
        large_workspace(workspace, Q, chunks), units_there, A8, qscale, stride, K8, Bw, Sa, Sb, chunks, R, Q, scale_inv, R_total, out, bias, st);
}

// Tile choice.  The 128 x 128 tile moves the fewest operand bytes per MAC and is the fastest whenever its grid
// covers the 256 CUs (one workgroup per CU at a time) -- measured up to several rounds of 256.  A smaller grid
// leaves CUs idle that smaller tiles would use: a workgroup's time per half-chunk is about 1 : 0.63 : 0.35 : 0.31
// for 128 x 128 : 128 x 64 : 64 x 64 : 64 x 32, so take the least (rounds of 256 workgroups x time), the larger
// tile on a tie.  g_i8_tile forces a tile (tuning and tests).
int choose_i8_tile(int64_t R, int64_t Q, int64_t* cost_out) {
    const int64_t n128 = ((R + 127) / 128) * ((Q + 127) / 128);
    if (cost_out) *cost_out = ((n128 + 255) / 256) * 100;
    if (const int forced = g_i8_tile.load(std::memory_order_relaxed); forced != 0 && forced != kLargeTile) return forced;
    if (n128 > 256) return 128;
    const int64_t cost[4] = {100, ((((R + 127) / 128) * ((Q + 63) / 64) + 255) / 256) * 63,
                             ((((R + 63) / 64) * ((Q + 63) / 64) + 255) / 256) * 35,
                             ((((R + 63) / 64) * ((Q + 31) / 32) + 255) / 256) * 31};
    const int tiles[4] = {128, 12864, 64, 6432};
    int best = 0;
    for (int i = 1; i < 4; ++i)
        if (cost[i] < cost[best]) best = i;
    if (cost_out) *cost_out = cost[best];
    return tiles[best];
}

// Half a round over: three rounds of 128 x 64 for two, where rows are short enough for a tile's start and stores to count.  us a layer, 128
// x 128 and 128 x 64, 512 and 1024 wide: 768 x 8192 keys bf16 14.3, 13.5 and 17.7, 17.1; 1280 x 4096 f32 15.4, 14.5 and 18.9, 18.3; 3000 x
// 1920 bf16 15.2, 14.1 and 20.5, 18.8; 530 x 8192 f32 14.7, 13.5 and 17.3, 17.0 -- 2048 wide 768 x 8192 f32 25.2, 25.7, 1536 x 4096 bf16 26.2,
// 26.7; 256 wide 1280 x 4096 bf16 12.5, 11.5, but 768 x 8192 14.3, 16.1.  A dot, which streams its outputs out, from three chunks on: 640 x
// 1024 x 8192 14.4, 12.4; 768 x 512 x 8192 9.7, 10.2.
int choose_i8_chain_tile(int64_t R, int64_t Q, int chunks, bool layer) {
    const int tile = choose_i8_tile(R, Q);
    const int64_t n128 = ((R + 127) / 128) * ((Q + 127) / 128);
    if (tile != 128 || g_i8_tile.load(std::memory_order_relaxed) == 128 || n128 <= 256 || n128 > 384) return tile;
    return chunks >= (layer ? 2 : 3) && chunks <= 4 && ((R + 127) / 128) * ((Q + 63) / 64) <= 768 ? 12864 : tile;
}

void i8_launch_shape(int64_t Q, int64_t R, unsigned* groups, int* waves) {
    const int tile = choose_i8_tile(R, Q);
    const int64_t tm = tile == 64 || tile == 6432 ? 64 : 128, tn = tile == 6432 ? 32 : (tile == 64 || tile == 12864 ? 64 : 128);
    *groups = static_cast<unsigned>(((R + tm - 1) / tm) * ((Q + tn - 1) / tn));
    *waves = (tile == 64 ? I8Cfg<64, 64>::kBlock : tile == 6432 ? I8Cfg<64, 32>::kBlock : tile == 12864 ? I8Cfg<128, 64>::kBlock
                                                                                     : I8Cfg<128, 128>::kBlock) / 64;
}

// D-split choice for a chain-mode call whose grid leaves most CUs idle: the 128 x 128 or 128 x 64 tile with `segments`
// workgroups per tile over runs of chunks, if the calling thread has attached a scratch region that holds the
// partial sums and the modelled time beats the best unsplit tile.  The model, in microseconds, from measurements on
// the MI355X: a workgroup's half-chunk costs 0.0045 us per unit of choose_i8_tile's scale; the partial sums' way
// through memory (stores, one write-back fence per workgroup, the counter, the last workgroup's loads) costs about
// 2 + 0.9 x segments + 0.5 per MiB of partial sums.  That overhead is why shapes like Q512 x R2048 x D8192 stay
// unsplit (16.3 us on 64 x 64 tiles against 22.6 - 26.5 split), and why grids of a few tiles over long rows split
// (Q128 x R512 x D16384: 20.0 -> 13.6 us; Q64 x R256 x D32768: 37.0 -> 17.3; Q256 x R1024 x D16384: 24.9 -> 18.3).
// Returns the tile (128 or 12864) and sets *segments, or 0 for no split.  g_i8_split: 0 = by this model, 1 = never,
// n >= 2 = n segments on the forced tile (g_i8_tile 128 or 12864; 128 x 128 otherwise) whenever the scratch allows it.
thread_local unsigned char* t_split_scratch = nullptr;
thread_local size_t t_split_bytes = 0;
thread_local int t_split_device = -1;
std::atomic<int> g_i8_split{0};
constexpr double kCostUnitUs = 0.0045;
constexpr int kSplitMinChunks = 2;  // chunks per segment at least
constexpr int kSplitMaxSegments = 64;

static size_t split_scratch_need(int64_t tiles, int segments, int TM, int TN) {
    return kSplitCounterBytes + static_cast<size_t>(tiles) * segments * TM * TN * sizeof(float);
}

int choose_i8_split(int64_t R, int64_t Q, int chunks, int* segments) {
    *segments = 1;
    const int mode = g_i8_split.load(std::memory_order_relaxed);
    if (mode == 1 || t_split_scratch == nullptr) return 0;
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev != t_split_device) return 0;
    const int64_t kr = (R + 127) / 128;
    const int64_t tiles_of[2] = {kr * ((Q + 127) / 128), kr * ((Q + 63) / 64)};
    const int tile_id[2] = {128, 12864}, tn_of[2] = {128, 64}, unit[2] = {100, 63};
    if (mode >= 2) {
        const int forced = g_i8_tile.load(std::memory_order_relaxed);
        const int i = forced == 12864 ? 1 : 0;
        const int seg = mode < chunks ? mode : chunks;
        if (seg < 2 || tiles_of[i] > kSplitMaxTiles || split_scratch_need(tiles_of[i], seg, 128, tn_of[i]) > t_split_bytes) return 0;
        *segments = seg;
        return tile_id[i];
    }
    if (tiles_of[0] >= 128) return 0;  // half the GPU busy on the large tile: nothing to gain
    int64_t unsplit = 0;
    (void)choose_i8_tile(R, Q, &unsplit);
    double best_us = kCostUnitUs * static_cast<double>(unsplit) * chunks * 2;
    int best = 0;
    for (int i = 0; i < 2; ++i) {
        const int64_t n = tiles_of[i];
        if (n > 128) continue;
        int max_seg = static_cast<int>(256 / n);
        if (max_seg > kSplitMaxSegments) max_seg = kSplitMaxSegments;
        if (max_seg > chunks / kSplitMinChunks) max_seg = chunks / kSplitMinChunks;
        for (int seg = 2; seg <= max_seg; ++seg) {
            const size_t need = split_scratch_need(n, seg, 128, tn_of[i]);
            if (need > t_split_bytes) break;
            const int64_t run = (chunks + seg - 1) / seg;  // chunks of the longest segment
            const double us = kCostUnitUs * unit[i] * static_cast<double>(run) * 2 + 2.0 + 0.9 * seg +
                              0.5 * static_cast<double>(need - kSplitCounterBytes) / (1 << 20);
            if (us < best_us) {
                best_us = us;
                best = tile_id[i];
                *segments = seg;
            }
        }
    }
    return best;
}

void launch_mfma_i8(const int8_t* A8, const float* qscale, int stride, const int8_t* K8, const float* Bw, int Sb,
                           int chunks, int64_t R, int64_t Q, int down_shift, float scale_inv, int64_t R_total,
                           float* out, int32_t* chunk_ints, const float* bias, hipStream_t st, int key_tiled,
                           int ndig, long long dig_stride, const long long* key_indices) {
    const bool chain = ndig == 0 && chunk_ints == nullptr && t_coop == nullptr;
    if (chain) {
        int segments = 1;
        const int split_tile = choose_i8_split(R, Q, chunks, &segments);
        if (split_tile == 128) {
            (t_out_dtype != BSI_DTYPE_F32 ? &launch_mfma_i8_split<128, 128, true> : &launch_mfma_i8_split<128, 128, false>)(
                segments, t_split_scratch, A8, qscale, stride, K8, Bw, Sb, chunks, R, Q, down_shift, scale_inv, R_total, out, bias, st,
                key_tiled);
            return;
        }
        if (split_tile == 12864) {
            (t_out_dtype != BSI_DTYPE_F32 ? &launch_mfma_i8_split<128, 64, true> : &launch_mfma_i8_split<128, 64, false>)(
                segments, t_split_scratch, A8, qscale, stride, K8, Bw, Sb, chunks, R, Q, down_shift, scale_inv, R_total, out, bias, st,
                key_tiled);
            return;
        }
    }
    const int tile = chain ? choose_i8_chain_tile(R, Q, chunks, t_layer_output != 0) : choose_i8_tile(R, Q);
    if (tile == 1284 && ndig == 0 && t_coop == nullptr) {
        launch_mfma_i8w<4>(A8, qscale, stride, K8, Bw, Sb, chunks, R, Q, down_shift, scale_inv, R_total, out, chunk_ints, bias,
                           st, key_tiled);
        return;
    }
#define BSI_I8_ARGS ndig, dig_stride, key_indices, key_tiled, A8, qscale, stride, K8, Bw, Sb, chunks, R, Q, down_shift, scale_inv, R_total, out, chunk_ints, bias, st
    if (tile == 128 || tile == 1284) launch_mfma_i8_t<128, 128>(BSI_I8_ARGS);
    else if (tile == 12864) launch_mfma_i8_t<128, 64>(BSI_I8_ARGS);
    else if (tile == 64) launch_mfma_i8_t<64, 64>(BSI_I8_ARGS);
    else launch_mfma_i8_t<64, 32>(BSI_I8_ARGS);
#undef BSI_I8_ARGS
}

}  // namespace bsi

using namespace bsi;

extern "C" size_t bsi_hip_dot_digits_workspace_bytes(int64_t Q, int nq, int64_t R, int nk) {
    if (Q <= 0 || R <= 0 || nq <= 0 || nk <= 0) return 0;
    return static_cast<size_t>(nq) * static_cast<size_t>(Q) * static_cast<size_t>(nk) * static_cast<size_t>(R) * 4;
}

extern "C" int bsi_hip_dot_digits(const int8_t* A_digits, int nq, const float* Aw, int Sa, const int8_t* K_digits, int nk,
                                  int preshift, const float* Bw, int Sb, int W64, int64_t R, int64_t Q,
                                  const int64_t* key_indices, float scale_inv, int64_t R_total, const float* bias,
                                  float* out, void* workspace, size_t workspace_bytes, int k_tiled, void* stream) {
    BSI_REQUIRE(R >= 0 && Q >= 0 && W64 >= 1, "bad shape");
    BSI_REQUIRE(nq >= 1 && nq <= 10 && nk >= 1 && nk <= 10, "digit counts must be in [1, 10] (got %d, %d)", nq, nk);
    BSI_REQUIRE(k_tiled == 0 || nk == 1, "a tiled key image is a single digit");
    BSI_REQUIRE(Sa >= 1 && Sb >= 1 && preshift >= 0 && preshift <= 14, "bad slice counts or preshift");
    BSI_REQUIRE(R_total >= R, "R_total (%lld) < R (%lld)", static_cast<long long>(R_total), static_cast<long long>(R));
    // |sum| <= 256 chunks' worth of 128 * 128 per element: int32 holds D up to 2^17 elements
    BSI_REQUIRE(W64 <= 2048, "more than 2^17 elements per row could overflow the int32 sums (W64 = %d)", W64);
    if (R == 0 || Q == 0) return BSI_OK;
    BSI_REQUIRE(A_digits && Aw && K_digits && Bw && out, "null pointer");
    const int64_t Qd = static_cast<int64_t>(nq) * Q, Rd = static_cast<int64_t>(nk) * R;
    BSI_REQUIRE((Qd + 31) / 32 <= 65535, "too many query rows for one launch");
    hipStream_t st = as_stream(stream);
    const int chunks = (W64 + 3) / 4;
    const long long dig_stride = static_cast<long long>(Q) * chunks * 256;
    // One key digit: the query digits are put back together in the accumulator (shift by 7 between digits) and the
    // epilogue writes the floats -- if int32 holds sum_d |query value| |key digit|: query bits (Sa - 1 + preshift
    // when nq == 1, as the image is pre-shifted) + 7 key bits + log2(elements) <= 31, and the digit images lie
    // within reach of a 32-bit buffer offset.
    int log2_elems = 0;
    while ((1LL << log2_elems) < static_cast<long long>(chunks) * 256) ++log2_elems;
    const int qbits = (nq == 1) ? 7 : (Sa - 1);
    const int kbits = (preshift == 0 && Sb <= 7) ? (Sb - 1) : 7;
    const bool can_fold = nk == 1 && qbits + kbits + log2_elems <= 31 && static_cast<long long>(nq) * dig_stride < (1LL << 31);
    // folding runs nq times the chunks on the grid of Q rows; stacking runs the chunks once on the grid of nq Q rows
    // and then reads the int32 products back (about 3 us + 4 bytes per product at 4 TB/s; one cost unit of the tile
    // model is about 0.012 us per chunk)
    int64_t cost_fold = 0, cost_stack = 0;
    const int tile_fold = choose_i8_tile(R, Q, &cost_fold);
    const int tile_stack = choose_i8_tile(Rd, Qd, &cost_stack);
    // without the chain's epilogue to overlap, the 64-key tiles come out about 1.3 times their modelled cost
    const double us_fold = 0.012 * static_cast<double>(cost_fold) * chunks * nq * ((tile_fold == 64 || tile_fold == 6432) ? 1.3 : 1.0);
    const double us_stack = 0.012 * static_cast<double>(cost_stack) * chunks * ((tile_stack == 64 || tile_stack == 6432) ? 1.3 : 1.0) + 3.0 +
                            static_cast<double>(nq * nk + 1) * static_cast<double>(Q) * static_cast<double>(R) * 4.0 / 4.0e6;
    const int route = g_digits_route.load(std::memory_order_relaxed);
    const bool fold = route == 2 || (route == 0 && (nq == 1 || us_fold <= us_stack));
    if (can_fold && fold) {
        launch_mfma_i8(A_digits, Aw, Sa, K_digits, Bw, Sb, chunks, R, Q, preshift, scale_inv, R_total, out, nullptr, bias,
                       st, k_tiled, nq, dig_stride, reinterpret_cast<const long long*>(key_indices));
        BSI_LAUNCH_CHECK("dot_mfma_i8_kernel (int32 sum, digits recombined in the accumulator)");
        return BSI_OK;
    }
    const size_t need = bsi_hip_dot_digits_workspace_bytes(Q, nq, R, nk);
    BSI_REQUIRE(workspace != nullptr && workspace_bytes >= need, "workspace too small: %zu < %zu bytes", workspace_bytes,
                need);
    // else one int8 GEMM over the stacked digits: I[i Q + q, j R + r] = sum_d A_i[q, d] K_j[r, d]
    launch_mfma_i8(A_digits, Bw, 1, K_digits, Bw, 1, chunks, Rd, Qd, 0, 1.0f, Rd, nullptr,
                   reinterpret_cast<int32_t*>(workspace), nullptr, st, k_tiled, 1, 0, nullptr);
    BSI_LAUNCH_CHECK("dot_mfma_i8_kernel (int32 sum)");
    const int64_t total = Q * R;
    launch(digits_combine_kernel, dim3(static_cast<unsigned>((total + 255) / 256)), dim3(256), 0, st,
                       reinterpret_cast<const int*>(workspace), nq, nk, Q, R, preshift, Aw, Sa, Bw, Sb,
                       reinterpret_cast<const long long*>(key_indices), scale_inv, R_total, bias, out);
    BSI_LAUNCH_CHECK("digits_combine_kernel");
    return BSI_OK;
}

extern "C" int bsi_hip_probe_l2_to_lds(const void* buf, size_t bytes, int loader_pattern, double* bytes_per_s, void* stream) {
    BSI_REQUIRE(buf && bytes_per_s, "null pointer");
    constexpr size_t kRegion = 256 * 1024;
    constexpr int kRegions = 8, kPasses = 64;
    BSI_REQUIRE(bytes >= kRegion * kRegions, "the probe streams %zu bytes of the buffer", kRegion * kRegions);
    hipStream_t st = as_stream(stream);
    int dev = 0, cus = 0;
    BSI_HIP_CHECK(hipGetDevice(&dev));
    BSI_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    const int lds = kProbeLdsWaves * kProbeLdsSlots * 1024;
    BSI_REQUIRE(loader_pattern >= 0 && loader_pattern <= 3, "loader_pattern must be 0, 1, 2 or 3");
    static LdsOptIn once0, once1, once2, once3;
    lds_opt_in(once0, reinterpret_cast<const void*>(&probe_l2_lds_kernel<8, 12, false>), lds);
    lds_opt_in(once1, reinterpret_cast<const void*>(&probe_l2_lds_kernel<4, 24, true>), lds);
    lds_opt_in(once2, reinterpret_cast<const void*>(&probe_l2_lds_kernel<4, 24, false>), lds);
    lds_opt_in(once3, reinterpret_cast<const void*>(&probe_l2_lds_kernel<8, 12, true>), lds);
    hipEvent_t e0, e1;
    BSI_HIP_CHECK(hipEventCreate(&e0));
    if (hipError_t ec = hipEventCreate(&e1); ec != hipSuccess) {
        (void)hipEventDestroy(e0);
        return fail(BSI_ERR_HIP, "hipEventCreate failed: %s", hipGetErrorString(ec));
    }
    float best = 1e30f;
    hipError_t err = hipSuccess;
    for (int rep = 0; rep < 4 && err == hipSuccess; ++rep) {  // the first repetition also brings the regions into L2
        (void)hipEventRecord(e0, st);
        if (loader_pattern == 1)
            launch((probe_l2_lds_kernel<4, 24, true>), dim3(static_cast<unsigned>(cus)), dim3(4 * 64), lds, st,
                               static_cast<const unsigned char*>(buf), kRegion, kRegions, kPasses);
        else if (loader_pattern == 2)
            launch((probe_l2_lds_kernel<4, 24, false>), dim3(static_cast<unsigned>(cus)), dim3(4 * 64), lds, st,
                               static_cast<const unsigned char*>(buf), kRegion, kRegions, kPasses);
        else if (loader_pattern == 3)
            launch((probe_l2_lds_kernel<8, 12, true>), dim3(static_cast<unsigned>(cus)), dim3(8 * 64), lds, st,
                               static_cast<const unsigned char*>(buf), kRegion, kRegions, kPasses);
        else
            launch((probe_l2_lds_kernel<8, 12, false>), dim3(static_cast<unsigned>(cus)), dim3(8 * 64), lds, st,
                               static_cast<const unsigned char*>(buf), kRegion, kRegions, kPasses);
        (void)hipEventRecord(e1, st);
        err = hipEventSynchronize(e1);
        float ms = 0.0f;
        if (err == hipSuccess) err = hipEventElapsedTime(&ms, e0, e1);
        if (rep > 0 && ms < best) best = ms;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (err != hipSuccess) return fail(BSI_ERR_HIP, "probe timing failed: %s", hipGetErrorString(err));
    BSI_LAUNCH_CHECK("probe_l2_lds_kernel");
    *bytes_per_s = static_cast<double>(cus) * kRegion * kPasses / (best * 1e-3);
    return BSI_OK;
}

extern "C" int bsi_hip_timeline_read(unsigned long long* stamps_host, int workgroups) {
    BSI_REQUIRE(stamps_host && workgroups >= 1 && workgroups <= kTimelineWorkgroups, "workgroups must be 1 .. %d",
                kTimelineWorkgroups);
#ifdef BSI_TIMELINE
    BSI_HIP_CHECK(hipDeviceSynchronize());
    BSI_HIP_CHECK(hipMemcpyFromSymbol(stamps_host, HIP_SYMBOL(g_timeline), sizeof(unsigned long long) * 8 * workgroups));
    void* dev = nullptr;  // cleared, so that the next read shows which workgroups have run since
    BSI_HIP_CHECK(hipGetSymbolAddress(&dev, HIP_SYMBOL(g_timeline)));
    BSI_HIP_CHECK(hipMemset(dev, 0, sizeof(unsigned long long) * 8 * kTimelineWorkgroups));
    return BSI_OK;
#else
    return fail(BSI_ERR_INVALID, "this library was built without the timeline stamps (make TIMELINE=1 builds one with)");
#endif
}

extern "C" int bsi_hip_timeline_read_cycles(unsigned long long* cycles_host, int workgroups) {
    BSI_REQUIRE(cycles_host && workgroups >= 1 && workgroups <= kTimelineWorkgroups, "workgroups must be 1 .. %d",
                kTimelineWorkgroups);
#ifdef BSI_TIMELINE
    BSI_HIP_CHECK(hipDeviceSynchronize());
    BSI_HIP_CHECK(hipMemcpyFromSymbol(cycles_host, HIP_SYMBOL(g_timeline_cycles), sizeof(unsigned long long) * 8 * workgroups));
    return BSI_OK;
#else
    return fail(BSI_ERR_INVALID, "this library was built without the timeline stamps (make TIMELINE=1 builds one with)");
#endif
}
