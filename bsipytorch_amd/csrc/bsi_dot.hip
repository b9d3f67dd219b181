// Fixed-bit weighted-popcount dot for gfx950:  out[q,r] = scale_inv * sum_c  I[q,r,c] * qscale[q,c] * bscale[r]
// with I[q,r,c] = sum_{i,j} +-(popc(A_i & B_j over chunk c) << (i+j)) -- which is exactly the integer
// dot product of the two's-complement values the planes encode.  Two cores compute I:
//
//   VALU  v_and_b32 + v_bcnt_u32_b32 on bit-planes.  A 64x64 output tile per workgroup, key and
//         query plane tiles of one 256-element chunk staged in LDS, 4x4 outputs per lane, the key
//         planes of a half chunk held in VGPRs while the query planes stream through.
//   MFMA  planes are recombined to int8 (value << (8 - S), so the two's-complement sign bit lands on
//         the int8 sign bit) by an 8x8 bit-matrix transpose in registers, then
//         v_mfma_i32_16x16x64_i8 accumulates 2^(16-Sa-Sb) * I per chunk.  Keys are the M operand,
//         queries the N operand, so a lane owns one query column: its chunk scale is one value.
//
//         Kernels of this core, chosen by bsi_hip_dot from the key layout and the number of query rows:
//           dot_mfma_i8_kernel       compute-bound calls on the cached int8 image of the keys
//           dot_mfma_stream_kernel   a few query rows: streams the packed planes once (bandwidth-bound)
//           dot_mfma_stream_ewah_kernel   the same for one query handed over as EWAH streams
//           dot_mfma_ws_kernel       many rows on tiled planes (producer waves recombine the planes)
//           dot_mfma_kernel          canonical planes or slice counts other than 6
//
// Shapes in the comments are rows x width x keys.
//
// Operands whose slice count follows the data (decimal mode) carry float slice weights instead of scales:
//   dot_weighted_kernel      popcounts per slice pair, summed exactly in float64 (any Sa, Sb <= 64)
//   dot_mfma_i8_kernel in its int32-sum mode on int8 digit images (planes_to_digits_kernel), the digits put back
//   together in the accumulator or by digits_combine_kernel: the same sum on the matrix cores
//
// Both feed the same fp32 epilogue, in chunk order:  acc = fmaf((float)I, qscale[q,c], acc), then
// out = (acc * bscale[r]) * scale_inv.  bscale is a power of two, so hoisting it out of the chain is
// exact and the result is bit-identical to fmaf((float)I, qscale*bscale, acc) of the reference
// kernel (bsi_ops/csrc/cuda/bsi_cuda_kernels_dot.cuh:1447-1540).
//
// This file: validation, kernel selection and the entry points of the fixed-bit dot.  The kernels live by family in
// bsi_dot_i8.hip (int8 image of the keys), bsi_dot_few_rows.hip (a few query rows, planes streamed once),
// bsi_dot_planes.hip (many rows on planes), bsi_dot_valu.hip (popcount cores, weighted slices, bias) and
// bsi_dot_layouts.hip (operand layouts); bsi_dot_device.h holds the device helpers they share.
#include "bsi_coop_build.h"
#include "bsi_dot_internal.h"

namespace bsi {
static std::atomic<int> g_coop_patience{kCoopPatience}, g_coop_shares{0};
}  // namespace bsi

using namespace bsi;

extern "C" int bsi_hip_set_option(int option, int value) {
    switch (option) {
        case BSI_OPT_DIGITS_ROUTE:
            BSI_REQUIRE(value >= 0 && value <= 2, "route must be 0, 1 or 2");
            g_digits_route = value;
            return BSI_OK;
        case BSI_OPT_I8_TILE:
            BSI_REQUIRE(value == 0 || value == 128 || value == 1284 || value == 12864 || value == 64 || value == 6432 || value == 256,
                        "tile must be 0, 128, 1284, 12864, 64, 6432 or 256");
            g_i8_tile = value;
            return BSI_OK;
        case BSI_OPT_OUTPUT_STORES:
            BSI_REQUIRE(value >= 0 && value <= 2, "output stores must be 0 (by entry point), 1 (plain) or 2 (nontemporal)");
            g_output_stores = value;
            return BSI_OK;
        case BSI_OPT_I8_SPLIT:
            BSI_REQUIRE(value >= 0 && value <= 64, "split must be 0 (by cost), 1 (never) or a number of segments up to 64");
            g_i8_split = value;
            return BSI_OK;
        case BSI_OPT_COOP_PATIENCE:
            BSI_REQUIRE(value >= 0, "patience must not be negative");
            g_coop_patience = value;
            return BSI_OK;
        case BSI_OPT_COOP_SHARES:
            BSI_REQUIRE(value >= 0 && value <= kCoopShares, "shares must be 0 (by the launch) to %d", kCoopShares);
            g_coop_shares = value;
            return BSI_OK;
        case BSI_OPT_BUILD_ITEMS:
            BSI_REQUIRE(value == 0 || value == 1 || value == 2 || value == 4 || value == 8, "items must be 0, 1, 2, 4 or 8");
            g_build_items = value;
            return BSI_OK;
        default:
            return fail(BSI_ERR_INVALID, "unknown option %d", option);
    }
}

extern "C" size_t bsi_hip_dot_workspace_bytes(int64_t Q, int W64, int core) {
    if (core == BSI_CORE_VALU || Q <= 0 || W64 <= 0) return 0;
    return static_cast<size_t>(Q) * static_cast<size_t>((W64 + 3) / 4) * 256;
}

extern "C" size_t bsi_hip_dot_split_scratch_bytes(void) {
    // one round of 256 workgroups, each with the partial sums of a 128 x 128 tile
    return kSplitCounterBytes + static_cast<size_t>(256) * 128 * 128 * sizeof(float);
}

extern "C" int bsi_hip_dot_attach_split_scratch(void* scratch_device, size_t bytes) {
    if (scratch_device == nullptr || bytes == 0) {
        t_split_scratch = nullptr;
        t_split_bytes = 0;
        t_split_device = -1;
        return BSI_OK;
    }
    BSI_REQUIRE((reinterpret_cast<uintptr_t>(scratch_device) & 255) == 0, "the split scratch must be 256-byte aligned");
    BSI_REQUIRE(bytes > kSplitCounterBytes, "a split scratch holds %zu bytes of counters and then the partial sums (got %zu bytes)",
                kSplitCounterBytes, bytes);
    int dev = -1;
    BSI_HIP_CHECK(hipGetDevice(&dev));
    t_split_scratch = static_cast<unsigned char*>(scratch_device);
    t_split_bytes = bytes;
    t_split_device = dev;
    return BSI_OK;
}

extern "C" int bsi_hip_dot_split_plan(int64_t R, int64_t Q, int W64, int* tile, int* segments) {
    BSI_REQUIRE(tile && segments && R >= 1 && Q >= 1 && W64 >= 1, "bad arguments");
    const int split_tile = choose_i8_split(R, Q, (W64 + 3) / 4, segments);
    *tile = split_tile != 0 ? split_tile : choose_i8_chain_tile(R, Q, (W64 + 3) / 4, false);
    return BSI_OK;
}

// The matrix-core kernels address a tile's operand rows with 32-bit buffer offsets inside a descriptor of at most
// 2 GiB: 128 rows of chunks * 256 bytes must stay below that.
constexpr int kMfmaMaxChunks = 32768;

// What every route of the fixed-bit dot asks of its operands; BSI_OK where there is nothing to do.
static int check_dot(const uint64_t* A, const int8_t* A_ints8, const float* A_chunk_scales, int A_scale_stride, int Sa, int W64,
                     const uint64_t* B, int b_layout, const float* Bw, int Sb, int64_t R, int64_t Q, int64_t R_total, const void* out) {
    BSI_REQUIRE(Q >= 0 && R >= 0, "negative Q or R");
    BSI_REQUIRE(W64 >= 1, "W64 must be >= 1");
    BSI_REQUIRE(Sa >= 1 && Sa <= 63 && Sb >= 1 && Sb <= 63, "Sa and Sb must be in [1, 63]");
    BSI_REQUIRE(R_total >= R, "R_total must be >= R");
    // per-row operands (slice weights, bias, chunk scales) are fetched with 32-bit byte offsets
    BSI_REQUIRE(R <= (1 << 25) && Q <= (1 << 25), "at most 2^25 key rows and query rows per call (got R = %lld, Q = %lld)",
                static_cast<long long>(R), static_cast<long long>(Q));
    // query tiles (32 rows in the smallest kernel tile) ride on the launch grid's second dimension, which holds 65535
    BSI_REQUIRE((Q + 31) / 32 <= 65535, "at most 65535 x 32 query rows per call (got Q = %lld); split the batch",
                static_cast<long long>(Q));
    BSI_REQUIRE(b_layout == BSI_LAYOUT_CANONICAL || b_layout == BSI_LAYOUT_TILED16 || b_layout == BSI_LAYOUT_INT8 ||
                    b_layout == BSI_LAYOUT_INT8_TILED,
                "unknown key layout %d", b_layout);
    if (Q == 0 || R == 0) return BSI_OK;
    const int chunks = (W64 + 3) / 4;
    BSI_REQUIRE(A_chunk_scales != nullptr, "A_chunk_scales is required (pass a [Q,1] array of row scales if there are no chunk scales)");
    BSI_REQUIRE(A_scale_stride == chunks || A_scale_stride == 1,
                "chunk scale stride mismatch: got %d expected %d (or 1 for row scales)", A_scale_stride, chunks);
    BSI_REQUIRE(B && Bw && out, "null pointer");
    BSI_REQUIRE(A || A_ints8, "neither query planes nor int8 queries given");
    return BSI_OK;
}

// Validation, kernel selection and launch.  `bias` (optional) is added to every output; *bias_fused tells
// the caller whether the selected kernel did that in its own epilogue.
static int dot_launch(const uint64_t* A, const int8_t* A_ints8, const float* A_chunk_scales, int A_scale_stride,
                      int Sa, int W64, const uint64_t* B, int b_layout, const float* Bw, int Sb, int64_t R, int64_t Q,
                      float scale_inv, int64_t R_total, float* out, int32_t* chunk_ints, int core, void* workspace,
                      size_t workspace_bytes, void* stream, const float* bias, bool* bias_fused) {
    *bias_fused = false;
    if (int rc = check_dot(A, A_ints8, A_chunk_scales, A_scale_stride, Sa, W64, B, b_layout, Bw, Sb, R, Q, R_total, out)) return rc;
    if (Q == 0 || R == 0) return BSI_OK;
    const int chunks = (W64 + 3) / 4;
    hipStream_t st = as_stream(stream);

    const bool mfma_ok = (Sa >= 2 && Sa <= 8 && Sb >= 2 && Sb <= 8);
    if (core == BSI_CORE_AUTO) core = (mfma_ok && chunks <= kMfmaMaxChunks) ? BSI_CORE_MFMA : BSI_CORE_VALU;

    if (core == BSI_CORE_MFMA) {
        if (!mfma_ok) return fail(BSI_ERR_UNSUPPORTED, "MFMA core needs Sa, Sb in [2, 8] (got %d, %d)", Sa, Sb);
        if (chunks > kMfmaMaxChunks)
            return fail(BSI_ERR_UNSUPPORTED, "MFMA core takes rows of up to %d chunks of 256 elements (got %d)", kMfmaMaxChunks, chunks);
        const int8_t* A8 = A_ints8;
        BSI_REQUIRE((reinterpret_cast<uintptr_t>(A8) & 15) == 0 && (reinterpret_cast<uintptr_t>(workspace) & 15) == 0,
                    "int8 queries / workspace must be 16-byte aligned");
        if (A8 == nullptr) {
            const size_t need = bsi_hip_dot_workspace_bytes(Q, W64, core);
            BSI_REQUIRE(workspace != nullptr && workspace_bytes >= need,
                        "MFMA core without int8 queries needs %zu bytes of workspace (got %zu)", need, workspace_bytes);
            if (int rc = launch_planes_to_int8(A, Q, Sa, W64, static_cast<int8_t*>(workspace), st)) return rc;
            A8 = static_cast<const int8_t*>(workspace);
        }
        const int down_shift = 16 - Sa - Sb;
        if (b_layout == BSI_LAYOUT_INT8 || b_layout == BSI_LAYOUT_INT8_TILED) {
            BSI_REQUIRE((reinterpret_cast<uintptr_t>(B) & 15) == 0, "int8 key image must be 16-byte aligned");
            launch_mfma_i8(A8, A_chunk_scales, A_scale_stride, reinterpret_cast<const int8_t*>(B), Bw, Sb, chunks, R, Q,
                           down_shift, scale_inv, R_total, out, chunk_ints, bias, st,
                           b_layout == BSI_LAYOUT_INT8_TILED ? 1 : 0);
            BSI_LAUNCH_CHECK("dot_mfma_i8_kernel");
            *bias_fused = true;
            return BSI_OK;
        }
        const bool tiled = (b_layout == BSI_LAYOUT_TILED16);
        if (Sb == 6 && tiled && Q <= kStreamMaxQ) {
            launch_mfma_stream_by_shape(A8, A_chunk_scales, A_scale_stride, B, Bw, chunks, R, Q, down_shift, scale_inv, R_total,
                                        out, chunk_ints, bias, st);
            BSI_LAUNCH_CHECK("dot_mfma_stream_kernel");
            *bias_fused = true;
            return BSI_OK;
        }
        if (t_out_dtype != BSI_DTYPE_F32)
            return fail(BSI_ERR_UNSUPPORTED, "half-precision output: the kernels on key planes for many rows write float32 only");
        const char* kernel = launch_mfma_planes(tiled, A8, A_chunk_scales, A_scale_stride, B, Bw, Sb, W64, chunks, R, Q,
                                                down_shift, scale_inv, R_total, out, chunk_ints, st);
        BSI_LAUNCH_CHECK(kernel);
        return BSI_OK;
    }

    if (core != BSI_CORE_VALU) return fail(BSI_ERR_INVALID, "unknown core %d", core);
    if (b_layout == BSI_LAYOUT_INT8 || b_layout == BSI_LAYOUT_INT8_TILED)
        return fail(BSI_ERR_UNSUPPORTED, "the popcount core reads key planes, not the int8 image");
    BSI_REQUIRE(A != nullptr, "VALU core needs the query planes");
    if (t_out_dtype != BSI_DTYPE_F32) return fail(BSI_ERR_UNSUPPORTED, "half-precision output: the popcount core writes float32 only");
    if (Sa == 7 && Sb == 6) {
        launch_valu76(b_layout == BSI_LAYOUT_TILED16, A, A_chunk_scales, A_scale_stride, B, Bw, W64, chunks, R, Q, scale_inv,
                      R_total, out, chunk_ints, st);
        BSI_LAUNCH_CHECK("dot_valu_kernel");
        return BSI_OK;
    }
    const int64_t total = Q * R;
    BSI_REQUIRE((total + 255) / 256 <= 0x7fffffffLL, "too many outputs for one launch of the any-width kernel");
    launch_valu_generic(A, A_chunk_scales, A_scale_stride, Sa, B, Bw, Sb, W64, chunks, R, Q, scale_inv, R_total, out,
                        chunk_ints, b_layout == BSI_LAYOUT_TILED16 ? 1 : 0, st);
    BSI_LAUNCH_CHECK("dot_valu_generic_kernel");
    return BSI_OK;
}

namespace bsi {

int dot_with_bias(const uint64_t* A, const int8_t* A_ints8, const float* A_chunk_scales, int A_scale_stride,
                         int Sa, int W64, const uint64_t* B, int b_layout, const float* Bw, int Sb, int64_t R, int64_t Q,
                         float scale_inv, int64_t R_total, float* out, int32_t* chunk_ints, int core, void* workspace,
                         size_t workspace_bytes, void* stream, const float* bias) {
    bool fused = false;
    const int rc = dot_launch(A, A_ints8, A_chunk_scales, A_scale_stride, Sa, W64, B, b_layout, Bw, Sb, R, Q, scale_inv,
                              R_total, out, chunk_ints, core, workspace, workspace_bytes, stream, bias, &fused);
    if (rc != BSI_OK || bias == nullptr || fused || Q == 0 || R == 0) return rc;
    launch_add_bias(out, bias, Q, R, R_total, as_stream(stream));
    BSI_LAUNCH_CHECK("add_bias_kernel");
    return BSI_OK;
}

}  // namespace bsi

extern "C" int bsi_hip_dot(const uint64_t* A, const int8_t* A_ints8, const float* A_chunk_scales, int A_scale_stride,
                           int Sa, int W64, const uint64_t* B, int b_layout, const float* Bw, int Sb, int64_t R,
                           int64_t Q, float scale_inv, int64_t R_total, float* out, int32_t* chunk_ints, int core,
                           void* workspace, size_t workspace_bytes, void* stream) {
    return dot_with_bias(A, A_ints8, A_chunk_scales, A_scale_stride, Sa, W64, B, b_layout, Bw, Sb, R, Q, scale_inv,
                         R_total, out, chunk_ints, core, workspace, workspace_bytes, stream, nullptr);
}

extern "C" int bsi_hip_dot_bias(const uint64_t* A, const int8_t* A_ints8, const float* A_chunk_scales,
                                int A_scale_stride, int Sa, int W64, const uint64_t* B, int b_layout, const float* Bw,
                                int Sb, int64_t R, int64_t Q, float scale_inv, int64_t R_total, const float* bias,
                                float* out, int core, void* workspace, size_t workspace_bytes, void* stream) {
    t_layer_output = 1;
    const int rc = dot_with_bias(A, A_ints8, A_chunk_scales, A_scale_stride, Sa, W64, B, b_layout, Bw, Sb, R, Q, scale_inv,
                                 R_total, out, nullptr, core, workspace, workspace_bytes, stream, bias);
    t_layer_output = 0;
    return rc;
}

extern "C" int bsi_hip_dot_bias_warm(const uint64_t* A, const int8_t* A_ints8, const float* A_chunk_scales,
                                     int A_scale_stride, int Sa, int W64, const uint64_t* B, int b_layout, const float* Bw,
                                     int Sb, int64_t R, int64_t Q, float scale_inv, int64_t R_total, const float* bias,
                                     float* out, int core, void* workspace, size_t workspace_bytes, const void* warm,
                                     size_t warm_bytes, void* stream) {
    BSI_REQUIRE(warm != nullptr || warm_bytes == 0, "null warm-up region");
    g_warm_ptr = warm;
    g_warm_bytes = warm_bytes;
    t_layer_output = 1;
    const int rc = dot_with_bias(A, A_ints8, A_chunk_scales, A_scale_stride, Sa, W64, B, b_layout, Bw, Sb, R, Q, scale_inv,
                                 R_total, out, nullptr, core, workspace, workspace_bytes, stream, bias);
    g_warm_ptr = nullptr;
    g_warm_bytes = 0;
    t_layer_output = 0;
    return rc;
}

// ------------------------------------------------------------------ the dot without any allocation
// The int8 query operands that bsi_hip_dot derives into a caller's workspace go, here, into an array that is part
// of the library's device image: one copy per GPU, there from the moment the code object is loaded until the
// process ends.  In host code the array's name is only a handle for hipGetSymbolAddress; the device address it
// returns (one per device) is what the kernels get.
constexpr size_t kStaticScratchBytes = BSI_STATIC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];
static std::atomic<void*> g_scratch_ptr[64];  // per device: the array's address there, once looked up

static int static_scratch(void** out) {
    int dev = 0;
    BSI_HIP_CHECK(hipGetDevice(&dev));
    BSI_REQUIRE(dev >= 0 && dev < 64, "device index %d is beyond the 64 this entry point keeps addresses for", dev);
    void* p = g_scratch_ptr[dev].load(std::memory_order_acquire);
    if (p == nullptr) {
        BSI_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        BSI_REQUIRE(p != nullptr, "hipGetSymbolAddress returned no address for the scratch array");
        g_scratch_ptr[dev].store(p, std::memory_order_release);
    }
    *out = p;
    return BSI_OK;
}

extern "C" int bsi_hip_dot_static_scratch(const uint64_t* A, const float* A_chunk_scales, int A_scale_stride, int Sa,
                                          int W64, const uint64_t* B, int b_layout, const float* Bw, int Sb, int64_t R,
                                          int64_t Q, float scale_inv, int64_t R_total, float* out, int32_t* chunk_ints,
                                          void* stream) {
    BSI_REQUIRE(A != nullptr, "the query planes are required (the int8 operands are derived from them)");
    BSI_REQUIRE(Sa >= 2 && Sa <= 8 && Sb >= 2 && Sb <= 8, "the matrix-core dot needs Sa, Sb in [2, 8] (got %d, %d)", Sa, Sb);
    BSI_REQUIRE(Q >= 0 && W64 >= 1, "bad shape");
    const size_t need = bsi_hip_dot_workspace_bytes(Q, W64, BSI_CORE_MFMA);
    BSI_REQUIRE(need <= kStaticScratchBytes,
                "Q x padded D = %zu bytes of int8 query operands exceed the %zu-byte static scratch; use bsi_hip_dot "
                "with a workspace", need, kStaticScratchBytes);
    void* ws = nullptr;
    if (int rc = static_scratch(&ws)) return rc;
    return dot_with_bias(A, nullptr, A_chunk_scales, A_scale_stride, Sa, W64, B, b_layout, Bw, Sb, R, Q, scale_inv, R_total,
                         out, chunk_ints, BSI_CORE_MFMA, ws, kStaticScratchBytes, stream, nullptr);
}

// Workspace of bsi_hip_linear: the query operands of one build (planes, shifts, scales, int8 image), each 256-aligned.
struct LinearWorkspace {
    size_t words, shifts, scales, ints8, large, total;  // large: where what the integer sums of a large layer take begins
};
static LinearWorkspace linear_workspace(int64_t Q, int64_t d, int fixed_bits) {
    const size_t W = static_cast<size_t>((d + 63) / 64), chunks = static_cast<size_t>((d + 255) / 256);
    auto up = [](size_t v) { return (v + 255) / 256 * 256; };
    LinearWorkspace w;
    w.words = 0;
    w.shifts = up(static_cast<size_t>(Q) * fixed_bits * W * 8);
    w.scales = w.shifts + up(static_cast<size_t>(Q) * chunks * 4);
    w.ints8 = w.scales + up(static_cast<size_t>(Q) * chunks * 4);
    w.large = w.ints8 + up(static_cast<size_t>(Q) * chunks * 256);
    w.total = w.large + i8_large_workspace_bytes(Q, static_cast<int>(chunks < (1 << 20) ? chunks : 1 << 20));
    return w;
}

extern "C" size_t bsi_hip_linear_workspace_bytes(int64_t Q, int64_t d, int fixed_bits) {
    if (Q <= 0 || d <= 0 || fixed_bits < 2 || fixed_bits > 8) return 0;
    return linear_workspace(Q, d, fixed_bits).total;
}

static bool linear_is_large(int64_t Q, int chunks, int b_layout, int Sb, int64_t R, int core) {
    return core == BSI_CORE_AUTO && b_layout == BSI_LAYOUT_INT8 && Sb >= 2 && Sb <= 8 && R > 0 && i8_large_serves(Q, R, chunks);
}

extern "C" size_t bsi_hip_linear_workspace_bytes_for(int64_t Q, int64_t d, int fixed_bits, int b_layout, int Sb, int64_t R, int core) {
    if (Q <= 0 || d <= 0 || fixed_bits < 2 || fixed_bits > 8) return 0;
    const LinearWorkspace w = linear_workspace(Q, d, fixed_bits);
    const int64_t chunks = (d + 255) / 256;
    return chunks <= kMfmaMaxChunks && linear_is_large(Q, static_cast<int>(chunks), b_layout, Sb, R, core) ? w.total : w.large;
}

extern "C" int bsi_hip_linear_plan(int64_t Q, int64_t d, int64_t R, int64_t R_total, int out_dtype, int* tile, int* streamed) {
    BSI_REQUIRE(tile && streamed && Q >= 1 && d >= 1 && R >= 1 && R_total >= R && d <= 256LL * kMfmaMaxChunks, "bad arguments");
    const int chunks = static_cast<int>((d + 255) / 256);
    int segments = 1;
    const int split_tile = choose_i8_split(R, Q, chunks, &segments);
    const bool large = i8_large_serves(Q, R, chunks);
    *tile = large ? kLargeTile : split_tile != 0 ? split_tile : choose_i8_chain_tile(R, Q, chunks, true);
    t_layer_output = 1;
    *streamed = out_dtype == BSI_DTYPE_F32 && R_total % 32 == 0 ? stream_output(R_total, Q, chunks) : 0;
    t_layer_output = 0;
    return BSI_OK;
}

extern "C" int bsi_hip_linear(const void* x, int dtype, int64_t Q, int64_t d, int decimal_places, int fixed_bits, int rebuild,
                              void* workspace, size_t workspace_bytes, const uint64_t* B, int b_layout, const float* Bw,
                              int Sb, int64_t R, float scale_inv, int64_t R_total, const float* bias, float* out, int core,
                              const void* warm, size_t warm_bytes, void* stream) {
    return bsi_hip_linear_out(x, dtype, Q, d, decimal_places, fixed_bits, rebuild, workspace, workspace_bytes, B, b_layout, Bw, Sb,
                              R, scale_inv, R_total, bias, out, BSI_DTYPE_F32, core, warm, warm_bytes, stream);
}

extern "C" int bsi_hip_linear_out(const void* x, int dtype, int64_t Q, int64_t d, int decimal_places, int fixed_bits, int rebuild,
                                  void* workspace, size_t workspace_bytes, const uint64_t* B, int b_layout, const float* Bw,
                                  int Sb, int64_t R, float scale_inv, int64_t R_total, const float* bias, void* out,
                                  int out_dtype, int core, const void* warm, size_t warm_bytes, void* stream) {
    BSI_REQUIRE(Q >= 0 && R >= 0 && d >= 1, "bad shape");
    BSI_REQUIRE(fixed_bits >= 2 && fixed_bits <= 8, "fixed_bits must be in [2, 8] (got %d)", fixed_bits);
    BSI_REQUIRE(out_dtype == BSI_DTYPE_F32 || out_dtype == BSI_DTYPE_F16 || out_dtype == BSI_DTYPE_BF16, "unknown dtype code %d", out_dtype);
    if (Q == 0 || R == 0) return BSI_OK;
    const int W64 = static_cast<int>((d + 63) / 64), chunks = (W64 + 3) / 4;
    const LinearWorkspace w = linear_workspace(Q, d, fixed_bits);
    BSI_REQUIRE(workspace != nullptr && workspace_bytes >= w.large, "workspace of %zu bytes needed, %zu given", w.large,
                workspace_bytes);
    BSI_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 255) == 0, "workspace must be 256-byte aligned");
    unsigned char* ws = static_cast<unsigned char*>(workspace);
    uint64_t* words = reinterpret_cast<uint64_t*>(ws + w.words);
    int32_t* shifts = reinterpret_cast<int32_t*>(ws + w.shifts);
    float* scales = reinterpret_cast<float*>(ws + w.scales);
    int8_t* ints8 = reinterpret_cast<int8_t*>(ws + w.ints8);
    const int chunk_scale = W64 % 4 == 0 ? 1 : 0;  // the builder's rule: else one scale per row
    // The matrix-core kernels read the int8 image only: the planes are built for the popcount core (asked for, or what
    // BSI_CORE_AUTO falls back to for wide keys), and where the builder cannot leave them out.
    const bool planes = core == BSI_CORE_VALU || Sb < 2 || Sb > 8 || chunks > kMfmaMaxChunks ||
                        integer_decimal_scale(pow(10.0, static_cast<double>(decimal_places))) == 0;
    BSI_REQUIRE(warm != nullptr || warm_bytes == 0, "null warm-up region");
    const bool large = workspace_bytes >= w.total && linear_is_large(Q, chunks, b_layout, Sb, R, core);
    if (large) {
        if (int rc = check_dot(nullptr, ints8, scales, chunk_scale ? chunks : 1, fixed_bits, W64, B, b_layout, Bw, Sb, R, Q, R_total, out)) return rc;
        BSI_REQUIRE((reinterpret_cast<uintptr_t>(B) & 15) == 0, "int8 key image must be 16-byte aligned");
    }
    const bool units_there = rebuild && large && chunk_scale && !planes;  // the units come out of the build
    if (units_there) {
        BSI_REQUIRE(dtype == BSI_DTYPE_F32 || dtype == BSI_DTYPE_F16 || dtype == BSI_DTYPE_BF16, "unknown dtype code %d", dtype);
        BSI_REQUIRE(x != nullptr, "null pointer");
        launch_build_units(ws + w.large, x, dtype, Q, d, fixed_bits, Sb, pow(10.0, static_cast<double>(decimal_places)), shifts, scales, ints8, chunks,
                           as_stream(stream));
        BSI_LAUNCH_CHECK("build_units_kernel");
    } else if (rebuild) {
        const int rc = bsi_hip_build_fixed(x, dtype, Q, d, decimal_places, fixed_bits, chunk_scale, 0.0f, planes ? words : nullptr,
                                           shifts, scales, ints8, stream);
        if (rc != BSI_OK) return rc;
    }
    t_out_dtype = out_dtype;
    if (large) {
        g_warm_ptr = warm;
        g_warm_bytes = warm_bytes;
        t_layer_output = 1;
        launch_i8_large(ws + w.large, units_there, ints8, scales, chunk_scale ? chunks : 1, reinterpret_cast<const int8_t*>(B), Bw, fixed_bits, Sb, chunks, R, Q,
                        scale_inv, R_total, static_cast<float*>(out), bias, as_stream(stream));
        g_warm_ptr = nullptr;
        g_warm_bytes = 0;
        t_layer_output = 0;
        t_out_dtype = BSI_DTYPE_F32;
        BSI_LAUNCH_CHECK("dot_mfma_i8_large_kernel");
        return BSI_OK;
    }
    const int rc = bsi_hip_dot_bias_warm(planes ? words : nullptr, ints8, scales, chunk_scale ? chunks : 1, fixed_bits, W64, B, b_layout,
                                         Bw, Sb, R, Q, scale_inv, R_total, bias, static_cast<float*>(out), core, nullptr, 0, warm,
                                         warm_bytes, stream);
    t_out_dtype = BSI_DTYPE_F32;
    return rc;
}

extern "C" size_t bsi_hip_linear_coop_bytes(void) { return kCoopBytes; }

// 0: not served; 1: a wave of the build takes a chunk at a time; 2: a whole row (kCoopHeld chunks at most)
static int coop_plan(int64_t Q, int64_t d, int64_t R, int decimal_places, int fixed_bits, int b_layout, int Sb) {
    const int64_t chunks = (d + 255) / 256;
    if (Q < 1 || d < 1 || R < 1 || Q * chunks > kCoopMaxItems || decimal_places < 0 || decimal_places > 2 || fixed_bits < 2 || fixed_bits > 8)
        return 0;
    unsigned groups = 0;
    int waves = 0;
    if (b_layout == BSI_LAYOUT_TILED16) {
        if (Q > kStreamMaxQ || Sb != 6) return 0;
        stream_launch_shape(Q, R, static_cast<int>(chunks), &groups, &waves);
    } else {
        if ((b_layout != BSI_LAYOUT_INT8 && b_layout != BSI_LAYOUT_INT8_TILED) || Sb < 2 || Sb > 8) return 0;
        i8_launch_shape(Q, R, &groups, &waves);
    }
    // Chunks that a wave of the build takes one after the other, each a load's latency: up to two chunk-scaled ones or one
    // of a row (which has barriers besides) cost less than a launch.  us a pass, two launches and one: 16 x 512 x 1280 6.6, 4.8;
    // 15 x 2560 x 5888 8.4, 7.3; 28 x 3072 x 4864 11.5, 10.6; 49 x 512 x 3328 6.9, 5.7; 121 x 512 x 14848 8.8, 8.1.
    const bool by_row = ((d + 63) / 64) % 4 != 0;
    CoopBuild b{};
    b.rows = static_cast<int>(Q);
    b.chunks = static_cast<int>(chunks);
    b.by_row = by_row ? 1 : 0;
    const int pieces = static_cast<int>(by_row ? Q : Q * chunks);
    if (by_row) {
        if (Q <= coop_shares(coop_groups(groups, R, b, waves), pieces) && chunks <= waves) return 1;
        b.row_per_wave = 1;
        const int shares = coop_shares(coop_groups(groups, R, b, waves), pieces);
        // A wave a row, for more rows: one load's latency too, but longer work and copies.  us, two launches (on a host that issues
        // them in 8.4, and on one that takes 9.8) and one: 24 x 704 x 704 8.4, 9.5, 6.6; 24 x 1600 x 1600 8.1, 9.5, 6.6; 100 x 320 x
        // 2000 8.5, 9.8, 6.8; 37 x 704 x 9728 8.5, 9.9, 7.0; 250 x 100 x 8192 8.7, 10.1, 7.6; 64 x 1600 x 4800 8.4, 9.8, 8.3; 77 x 1600 x
        // 4800 8.7, 9.9, 8.8 -- beyond: 121 x 1600 x 6400 (847 items) 8.9, 9.8, 9.7; 128 x 832 x 12000 (376 workgroups, whose registers
        // leave a CU one of them) 9.3, 9.9, 9.7.  Few tiles, with workgroups for the build beside them (-, the second host, one): 40 x 320 x 320
        // 9.7, 6.5; 200 x 704 x 704 9.4, 6.5; 500 x 320 x 320 9.6, 7.1; 128 x 1600 x 512 (896 items) 9.5, 8.0; 300 x 704 x 704 (900) 9.5, 7.0.
        // The edge at 560 items for more than 1024 keys, us in two launches on three hosts and in one: 539 items (77 x 1600 x 4800) 7.6, 8.8, 9.2,
        // 8.2; 560 (70 x 1984 x 4000) -, 9.2, 10.0, 8.6; beyond: 588 (84 x 1600 x 4800) 7.6, 8.7, 9.0, 8.2; 600 (150 x 960 x 4000) 7.1, 8.7, 9.0,
        // 8.1; 630 (90 x 1600 x 4800) 7.7, 8.7, 8.7, 8.4; 660 (220 x 704 x 6000) 9.2, -, 9.7, 10.0; 720 (120 x 1472 x 4096) 7.3, 8.6, 8.9, 8.2; 720
        // (90 x 1984 x 5000) 8.2, -, 8.8, 9.1; 728 (104 x 1600 x 4800) 8.1, 8.9, 9.1, 9.6; 784 (112 x 1600 x 4800) 8.1, -, 9.2, 9.6; 900 (300 x
        // 576 x 2048) 7.1, -, 8.9, 8.5.  One launch is bound by the GPU, two by the host: up to some 600 items it gains on most hosts and loses
        // at most half a microsecond on the fastest; from 730 on it loses on all.  Rows beyond 512: 500 x 192 x 2000 -, 9.0, 9.4, 7.9,
        // but 550 x 192 x 2000 -, 9.2, 9.3, 10.0 and 560 x 100 x 2000 -, 9.3, 9.5, 9.7.
        const int rounds = chunks <= 2 ? 3 : (chunks <= 4 ? 2 : 1);
        return Q <= 512 && Q <= rounds * static_cast<int64_t>(shares) * waves && chunks <= kCoopHeld && d % 4 == 0 &&
                       Q * chunks <= (R <= 1024 ? 1000 : 560) && groups <= 256
                   ? 2 : 0;
    }
    const int64_t items = Q * chunks, a_round = static_cast<int64_t>(coop_shares(coop_groups(groups, R, b, waves), pieces)) * waves;
    if (b_layout == BSI_LAYOUT_TILED16) {
        // us, two launches and one, with workgroups for the build where the tiles are few: 24 x 2304 x 256 9.3, 6.7; 32 x 2048 x 1024 9.1, 6.1;
        // 24 x 4096 x 512 9.0, 7.7; 32 x 4096 x 512 9.2, 7.8.
        return items <= 2 * a_round || (items <= 4 * a_round && items <= 512 && chunks <= 8) ? 1 : 0;
    }
    if (items <= 2 * static_cast<int64_t>(coop_shares(groups, pieces)) * waves) return 1;
    // More rounds: the launch takes some 3.75 us, 0.755 a round, 0.32 a chunk (each a step of the dot) and 1.9 for a million outputs, half a
    // microsecond more or less (64 sizes of 33 to 512 rows); two launches 8.3 to 8.8 on most hosts.  us, two launches there and one: 33 x 768 x
    // 768 8.6, 5.7; 256 x 768 x 768 8.4, 7.5; 333 x 768 x 768 8.5, 8.4; 128 x 1024 x 1024 8.5, 6.9; 200 x 1024 x 1024 8.5, 7.8; 100 x 1536 x 1536
    // 8.5, 7.7; 33 x 2048 x 2048 8.7, 7.0; 64 x 2048 x 2048 8.7, 8.2; 256 x 768 x 3072 8.5, 7.9 -- beyond: 128 x 1536 x 1536 8.6, 8.1; 256 x 1024 x
    // 1024 8.5, 8.7; 200 x 1024 x 4096 8.6, 8.4; 512 x 512 x 2048 8.5, 8.9; 100 x 2048 x 2048 8.6, 8.9; 333 x 768 x 3072 8.4, 9.2.  A host in its
    // fastest state issues two launches in 6.8: 256 x 512 x 512 6.8, 6.4; 333 x 512 x 512 6.8, 7.1; 512 x 512 x 512 6.8, 8.2.
    // Layers that are fed one tensor (q, k and v) share a build in two launches and not in one: three of them and nothing else, us, 33 x 768 x
    // 768 20.8, 17.2; 200 x 768 x 768 20.2, 20.1; 256 x 768 x 768 20.3, 21.6; 512 x 512 x 512 15.9, 22.7.  In a decoder, whose other kernels leave the GPU
    // waiting for the host, one launch still gains there: passes through three or four layers of 333 x 512 472, 432; 512 x 512 470, 442; 333 x 768
    // 356, 332; 200 x 1024 351, 327.  So the line lies where a single layer gains on most hosts.
    const double us = 0.755 * static_cast<double>(items) / static_cast<double>(a_round) + 0.32 * static_cast<double>(chunks) +
                      1.9e-6 * static_cast<double>(Q) * static_cast<double>(R);
    return groups <= 256 && us <= 4.4 ? 1 : 0;
}

extern "C" int bsi_hip_linear_coop_serves(int64_t Q, int64_t d, int64_t R, int decimal_places, int fixed_bits, int b_layout, int Sb) {
    return coop_plan(Q, d, R, decimal_places, fixed_bits, b_layout, Sb) != 0 ? 1 : 0;
}

extern "C" int bsi_hip_linear_coop_out(const void* x, int dtype, int64_t Q, int64_t d, int decimal_places, int fixed_bits, uint64_t launch_number,
                                       void* area, const uint64_t* B, int b_layout, const float* Bw, int Sb, int64_t R, float scale_inv,
                                       int64_t R_total, const float* bias, void* out, int out_dtype, const void* warm, size_t warm_bytes,
                                       void* stream) {
    BSI_REQUIRE(out_dtype == BSI_DTYPE_F32 || out_dtype == BSI_DTYPE_F16 || out_dtype == BSI_DTYPE_BF16, "unknown dtype code %d", out_dtype);
    BSI_REQUIRE(dtype == BSI_DTYPE_F32 || dtype == BSI_DTYPE_F16 || dtype == BSI_DTYPE_BF16, "unknown dtype code %d", dtype);
    const int plan = coop_plan(Q, d, R, decimal_places, fixed_bits, b_layout, Sb);
    if (plan == 0)
        return fail(BSI_ERR_UNSUPPORTED, "no launch with the query build inside for this layer");
    BSI_REQUIRE(x != nullptr && area != nullptr && launch_number != 0, "null pointer or launch number");
    BSI_REQUIRE((reinterpret_cast<uintptr_t>(area) & 255) == 0, "the area must be 256-byte aligned");
    const int W64 = static_cast<int>((d + 63) / 64), chunks = (W64 + 3) / 4;
    const double dec_scale = pow(10.0, static_cast<double>(decimal_places));
    const size_t esize = dtype == BSI_DTYPE_F32 ? 4 : 2;
    CoopBuild c{};
    c.x = x;
    c.area = static_cast<unsigned char*>(area);
    c.launch = launch_number;
    c.d = d;
    c.dec_scale = dec_scale;
    c.scale = static_cast<float>(dec_scale);
    c.dtype = dtype;
    c.vec = d % 4 == 0 && reinterpret_cast<uintptr_t>(x) % (4 * esize) == 0 ? 1 : 0;
    c.rows = static_cast<int>(Q);
    c.chunks = chunks;
    c.slices = fixed_bits;
    c.patience = g_coop_patience.load(std::memory_order_relaxed);
    c.shares = g_coop_shares.load(std::memory_order_relaxed);
    c.by_row = W64 % 4 == 0 ? 0 : 1;  // the builder's rule
    c.row_per_wave = plan == 2 ? 1 : 0;
    t_coop = &c;
    t_out_dtype = out_dtype;
    // the operands stand for the launch's own copies
    const int rc = bsi_hip_dot_bias_warm(nullptr, static_cast<const int8_t*>(area), static_cast<const float*>(area), c.by_row ? 1 : chunks,
                                         fixed_bits, W64, B, b_layout, Bw, Sb, R, Q, scale_inv, R_total, bias, static_cast<float*>(out),
                                         BSI_CORE_MFMA, nullptr, 0, warm, warm_bytes, stream);
    t_out_dtype = BSI_DTYPE_F32;
    t_coop = nullptr;
    return rc;
}

extern "C" int bsi_hip_dot_timed(const uint64_t* A, const int8_t* A_ints8, const float* A_chunk_scales,
                                 int A_scale_stride, int Sa, int W64, const uint64_t* B, int b_layout, const float* Bw,
                                 int Sb, int64_t R, int64_t Q, float scale_inv, int64_t R_total, float* out, int core,
                                 void* workspace, size_t workspace_bytes, int iters, float* mean_us, void* stream) {
    BSI_REQUIRE(iters >= 1 && mean_us, "iters must be >= 1 and mean_us non-null");
    hipStream_t st = as_stream(stream);
    hipEvent_t e0, e1;
    BSI_HIP_CHECK(hipEventCreate(&e0));
    if (hipError_t ec = hipEventCreate(&e1); ec != hipSuccess) {
        (void)hipEventDestroy(e0);
        return fail(BSI_ERR_HIP, "hipEventCreate failed: %s", hipGetErrorString(ec));
    }
    int rc = BSI_OK;
    hipError_t se = hipEventRecord(e0, st);
    for (int i = 0; i < iters && rc == BSI_OK; ++i)
        rc = bsi_hip_dot(A, A_ints8, A_chunk_scales, A_scale_stride, Sa, W64, B, b_layout, Bw, Sb, R, Q, scale_inv,
                         R_total, out, nullptr, core, workspace, workspace_bytes, stream);
    if (se == hipSuccess) se = hipEventRecord(e1, st);
    if (se == hipSuccess) se = hipEventSynchronize(e1);
    float ms = 0.0f;
    if (se == hipSuccess) se = hipEventElapsedTime(&ms, e0, e1);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc != BSI_OK) return rc;
    if (se != hipSuccess) return fail(BSI_ERR_HIP, "event timing failed: %s", hipGetErrorString(se));
    *mean_us = ms * 1000.0f / static_cast<float>(iters);
    return BSI_OK;
}
