// Device side of the EWAH encoder: the density flag and the one-wave encoder of a slice (the decoder, which the dot kernels
// use too, is ewah_expand_wave in bsi_common.h).
#pragma once
#include "bsi_common.h"

namespace bsi {

// 1 when a slice of W words with `count` set bits is to be run-length coded (bsi_cuda_kernels_ewah.cuh:35-69).
__device__ __forceinline__ int compress_flag(unsigned long long count, int W, double threshold) {
    const double total_bits = static_cast<double>(W) * 64.0;
    double p = (total_bits > 0.0) ? (static_cast<double>(count) / total_bits) : 0.0;
    if (p < 0.0) p = 0.0;
    if (p > 1.0) p = 1.0;
    // by squaring (0.1 us where two pow take over a microsecond); next to the threshold, where its rounding could matter, by pow
    double a = 1.0 - p, b = p;
#pragma unroll
    for (int i = 0; i < 7; ++i) {
        a *= a;
        b *= b;
    }
    double M = 1.0 - a - b;
    if (fabs(M - threshold) < 1.0e-9) M = 1.0 - pow(1.0 - p, 128.0) - pow(p, 128.0);
    return (M <= threshold) ? 1 : 0;
}

// One wave encodes one slice of W words (out == nullptr: size pass only).  Returns the stream length in every lane.
// The stream is the reference's greedy one (bsi_cuda_kernels_ewah.cuh:118-232): [marker: run of equal clean words,
// only when the slice is flagged][literals up to the next clean word] ..., an unflagged slice being one marker with
// W literals.  `first` is the lane's word of the first block (0 past the slice): a kernel that has other loads to wait for asks
// for it beside them.
__device__ __forceinline__ unsigned long long ewah_encode_wave(const unsigned long long* __restrict__ base, int W,
                                                               int compress, unsigned long long* __restrict__ out,
                                                               int lane, unsigned long long first) {
    const unsigned long long lt = (1ULL << lane) - 1ULL;  // lanes below this one
    unsigned long long n_starts = 0, n_lits = 0;          // markers / literal words before the current block
    // the segment that is open when a block begins: where it started, literals before it, its marker's place
    long long open_at = -1;
    unsigned long long open_lits = 0, open_pos = 0, open_bit = 0;
    unsigned long long prev_word = 0;
    bool prev_clean = false;
    for (int b = 0; b < W; b += BSI_WAVE) {
        const int i = b + lane;
        const bool valid = i < W;
        const unsigned long long v = b == 0 ? first : (valid ? base[i] : 0ULL);
        const bool clean = compress && valid && (v == 0ULL || v == ~0ULL);
        unsigned long long pv = __shfl_up(v, 1, BSI_WAVE);
        bool pc = __shfl_up(static_cast<int>(clean), 1, BSI_WAVE) != 0;
        if (lane == 0) {
            pv = prev_word;
            pc = prev_clean;
        }
        const bool start = valid && (i == 0 || (clean && (!pc || pv != v)));
        const bool lit = valid && !clean;
        const unsigned long long smask = __ballot(start), lmask = __ballot(lit), omask = __ballot(clean && v == ~0ULL);
        const unsigned long long starts_before = n_starts + __popcll(smask & lt);
        const unsigned long long lits_before = n_lits + __popcll(lmask & lt);
        if (out != nullptr) {
            if (lit) out[starts_before + (start ? 1ULL : 0ULL) + lits_before] = v;
            if (start && i > 0) {
                // this lane closes the segment before it: the nearest start below it in this block, else the open one
                const unsigned long long below = smask & lt;
                long long at;
                unsigned long long at_lits, at_pos, at_bit;
                if (below != 0ULL) {
                    const int L = 63 - __clzll(below);
                    const unsigned long long ltL = (1ULL << L) - 1ULL;
                    at = b + L;
                    at_lits = n_lits + __popcll(lmask & ltL);
                    at_pos = n_starts + __popcll(smask & ltL) + at_lits;
                    at_bit = (omask >> L) & 1ULL;
                } else {
                    at = open_at, at_lits = open_lits, at_pos = open_pos, at_bit = open_bit;
                }
                const unsigned long long seg_lits = lits_before - at_lits;
                const unsigned long long run_len = static_cast<unsigned long long>(i - at) - seg_lits;
                out[at_pos] = (run_len ? at_bit : 0ULL) | ((run_len & 0xFFFFFFFFULL) << 1) | (seg_lits << 33);
            }
        }
        if (smask != 0ULL) {  // the last start of this block is the open segment of the next one
            const int L = 63 - __clzll(smask);
            const unsigned long long ltL = (1ULL << L) - 1ULL;
            open_at = b + L;
            open_lits = n_lits + __popcll(lmask & ltL);
            open_pos = n_starts + __popcll(smask & ltL) + open_lits;
            open_bit = (omask >> L) & 1ULL;
        }
        n_starts += __popcll(smask);
        n_lits += __popcll(lmask);
        prev_word = __shfl(v, BSI_WAVE - 1, BSI_WAVE);
        prev_clean = __shfl(static_cast<int>(clean), BSI_WAVE - 1, BSI_WAVE) != 0;
    }
    if (out != nullptr && open_at >= 0 && lane == 0) {  // the last segment ends with the slice
        const unsigned long long seg_lits = n_lits - open_lits;
        const unsigned long long run_len = static_cast<unsigned long long>(W - open_at) - seg_lits;
        out[open_pos] = (run_len ? open_bit : 0ULL) | ((run_len & 0xFFFFFFFFULL) << 1) | (seg_lits << 33);
    }
    return n_starts + n_lits;
}
__device__ __forceinline__ unsigned long long ewah_encode_wave(const unsigned long long* __restrict__ base, int W, int compress,
                                                               unsigned long long* __restrict__ out, int lane) {
    return ewah_encode_wave(base, W, compress, out, lane, lane < W ? base[lane] : 0ULL);
}

}  // namespace bsi
