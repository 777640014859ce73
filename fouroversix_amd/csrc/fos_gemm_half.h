// Products with A converted ahead (fos_gemm_half.hip): its layout, the pass that produces it from codes and scales, the launch.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fos_gemm_common.h"
#include "fos_load_ranges.h"

namespace fos {

inline size_t fragment_bytes(int64_t rows, int64_t K) { return (size_t)((rows + 127) / 128) * (size_t)((K + 127) / 128) * kBandChunkBytes; }

// One operand, or two of the same inner dimension (rows 0: none).
struct ExpandOperand {
    const uint8_t *codes = nullptr, *sf = nullptr;
    uint8_t *out = nullptr;
    int64_t rows = 0;
};
struct ExpandParams {
    int64_t K, depth;  // K % 64 == 0; blocks from `depth` on are padding
    ExpandOperand operand[2];
    int groups = 0, groups_all = 0;  // blocks of 16 rows of the first one and of both (launch_expand_fragments)
};
int launch_expand_fragments(ExpandParams p, bool if4, hipStream_t s);

// Output tiles of the product: 256 x 256 (eight wavefronts), 128 x 256 and 128 x 128 (four); kHalfStream: up to 128 rows
// (NVFP4), the weight streamed once.
enum { kHalf256 = 1, kHalfWide, kHalfSmall, kHalfStream };
// p: frags, B, sfB (NVFP4), or frags and frags_b (IF4), ... ; with splits > 1 every split takes ksteps_per_split chunks of 128 k and the caller sums the partials.
int launch_gemm_half(GemmParams &p, int tile, bool if4, int out_type, hipStream_t s);

// The argument checks of an NVFP4 fos_gemm_linear_rows, nothing launched: for a caller that launches something ahead of it.
int check_gemm_linear(const uint8_t *A, const uint8_t *B, const uint8_t *sfA, const uint8_t *sfB, const float *amax_a, const float *amax_b,
                      double denominator, int64_t M, int64_t N, int64_t K, void *D, int out_type, int64_t ldd, const void *bias, float *d_amax);
// The product of a layer's call.  Its plan is made for fragments that the quantize kernel writes: linear_sizes says
// whether the shape takes them, at the beginning of the scratch, and how much of that there should be (`best`) or can be (`least`: from
// codes).  A null: they are there, otherwise codes and scales, for the
// same plan (`as_given`: an input that the streaming quantize kernels would read at another address) or for the one of
// products from codes.  Arguments checked by check_gemm_linear.
struct LinearSizes {
    size_t least, best;
    bool fragments;
};
LinearSizes linear_sizes(int64_t M, int64_t N, int64_t K);
int gemm_linear(const uint8_t *A, const uint8_t *B, const uint8_t *sfA, const uint8_t *sfB, const float *amax_a, const float *amax_b,
                double denominator, int64_t M, int64_t rows, int64_t N, int64_t K, void *D, int out_type, int64_t ldd, const void *bias,
                float *d_amax, bool as_given, void *scratch, size_t scratch_bytes, fos_stream_t stream);

// A layer's call for a few rows of bf16 input (contiguous, 16-byte aligned, cols % 16 == 0), quantization included, in one
// launch or, with K split, that and the reduction; kNotTaken where the shape is none for it.  In one launch d_amax has to be zero
// before (or an earlier maximum to extend).
constexpr int kNotTaken = 1;
bool linear_is_one_launch(int64_t M, int64_t N, int64_t K);
int gemm_decode_linear(const void *x, int64_t cols, int rule, const float *x_amax, const uint8_t *B, const uint8_t *sfB,
                       const float *amax_b, double denominator, int64_t M, int64_t N, int64_t K, void *D, int out_type, int64_t ldd,
                       const void *bias, float *d_amax, float *amax_word, void *partials, size_t partials_bytes, fos_stream_t stream);

}  // namespace fos
