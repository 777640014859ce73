// What the NVFP4 / IF4 products share: launch parameters, output scale, rounding of the outputs, recorded maximum, and
// the conversion of packed codes into fp16 operands.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fos_device.h"
#include "fouroversix_hip.h"

namespace fos {

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float16_t __attribute__((ext_vector_type(16)));
typedef float float4_t __attribute__((ext_vector_type(4)));

struct GemmParams {
    const uint8_t *A, *B;      // [M, K/2], [N, K/2]
    const uint8_t *sfA, *sfB;  // 128x4-tiled E4M3 bytes
    const uint8_t *frags, *frags_b;  // A, for IF4 B too, as fp16 fragments (fos_gemm_half.h), for the kernels that read them that way
    const float *alpha;        // output scale on the device, or null: (amax_a * amax_b) * inv_den
    const float *amax_a, *amax_b;
    float inv_den;
    int two_factors;           // an output scale outside fp32's normal range is applied in two factors (load_alpha)
    void *D;
    const void *bias;          // optional: N values of the output type, added to the rounded product and rounded again
    float *d_amax;             // optional: max|D| as stored is folded into d_amax[0] (unsigned atomic max on the bits)
    int64_t M, N, K, ldd;
    int64_t depth;             // columns of A and B from here on are padding (K % 64 == 0, K - depth < 64)
    uint32_t k_tail;           // IF4: mask on the scale bytes of the last 64 codes of a row, 0 for blocks that are padding
    int64_t cols;              // IF4: columns of D that exist, a multiple of 8 (the rest of N is padding that is not written)
    int64_t rows;              // rows 0 ... rows - 1 of D count for d_amax: padding rows hold the bias, not zeros
    int tiles_m, tiles_n;
    // split-K: workgroup (tile, blockIdx.y) contracts K steps [y * ksteps_per_split, ...) and
    // writes its FP32 partial tile to partials[y][M][N]; splits == 1 writes D directly
    float *partials;
    int splits, ksteps_per_split;
};

// Output scale: read from the device, or formed from the two tensor maxima with the
// arithmetic of gemm_alpha_kernel (product, then times the fp32 reciprocal of the divisor).
// `post`: with two_factors, what is left to multiply alpha * acc with (1 otherwise).  Maxima whose product, divided by
// the denominator, would be a sub-normal number with a few bits are multiplied 2^64 times too large; finite maxima
// whose product overflows, 2^64 times too small (with an infinite scale a sum of zero would become NaN and a small
// one infinite).  What still overflows then is a scale of 2^192 or more: any sum but zero, 2^-20 at least, is infinite
// with the largest number in its place too.
FOS_DEVICE float load_alpha(const GemmParams &p, float &post) {
    constexpr float kMax = 0x1.fffffep127f;
    post = 1.0f;
    if (p.alpha) return *p.alpha;
    const float a = *p.amax_a, b = *p.amax_b;
    if (p.two_factors && a * b < 0x1p-90f) {
        post = 0x1p-64f;
        return ((fminf(a, b) * 0x1p64f) * fmaxf(a, b)) * p.inv_den;
    }
    if (p.two_factors && a * b > kMax && a <= kMax && b <= kMax) {
        post = 0x1p64f;
        return fminf(((fmaxf(a, b) * 0x1p-64f) * fminf(a, b)) * p.inv_den, kMax);
    }
    return (a * b) * p.inv_den;
}

// Two values of the result as stored: rounded to the output type, packed in the low and the high half.
template <bool OUT_BF16>
FOS_DEVICE uint32_t round_pair(float v0, float v1) {
    if (OUT_BF16) {
        typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
        typedef float float2v __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, __builtin_convertvector((float2v{v0, v1}), bf16x2));
    }
    // (the values are products already rounded to fp32 -- the reference's epilogue multiplies in fp32, then converts -- and
    // must stay so: left to itself the compiler folds the multiplication into the conversion, v_fma_mixlo_f16,
    // which rounds the exact product once and differs from the two roundings in one output in 10^5)
    asm("" : "+v"(v0), "+v"(v1));
    return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)v0) | (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)v1) << 16;
}
template <bool OUT_BF16>
FOS_DEVICE float widen_out(uint32_t bits) {
    if (OUT_BF16) return u2f(bits << 16);
    return (float)__builtin_bit_cast(_Float16, (uint16_t)bits);
}

// Two consecutive outputs (columns n and n + 1, n % 2 == 0) from their scaled accumulators: rounded to the output
// type, and with a bias (its two values in `bias2`) rounded, added in fp32 and rounded again -- the two roundings of the
// reference's `out + bias` on the GEMM's result (src/fouroversix/model/modules/linear.py:83-92).  The magnitude
// bits of what is stored are folded into the halves of `umax` as unsigned 16-bit integers, which order finite
// values, infinity and NaN (largest) alike: a NaN in the output ends up as the recorded maximum, as it does
// in the reference's x.abs().max().  (Hardware conversions and packed maxima, 1.25 instructions per output after the
// multiplication by alpha, where rounding and maximum of each value in integer arithmetic took 7: whole layers of
// 16384 x 4096 -> 14336 1433 -> 1414 us, 1000 x 4096 -> 14336 104.1 -> 101.9, 2048 x 4096 -> 4096 71.9 -> 71.2.)
template <bool OUT_BF16>
FOS_DEVICE uint32_t finish_pair(float v0, float v1, bool with_bias, uint32_t bias2, uint32_t &umax) {
    typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
    uint32_t r = round_pair<OUT_BF16>(v0, v1);
    if (with_bias)
        r = round_pair<OUT_BF16>(widen_out<OUT_BF16>(r & 0xffffu) + widen_out<OUT_BF16>(bias2 & 0xffffu),
                                 widen_out<OUT_BF16>(r >> 16) + widen_out<OUT_BF16>(bias2 >> 16));
    umax = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, r & 0x7fff7fffu), __builtin_bit_cast(u16x2, umax)));
    return r;
}
// (maxima of two lots of outputs, as finish_pair forms them)
FOS_DEVICE uint32_t max_pairs(uint32_t a, uint32_t b) {
    typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b)));
}
// ... four (n % 4 == 0) and two consecutive outputs with the bias's values at n
template <bool OUT_BF16>
FOS_DEVICE uint2 pack_outputs(const float *v, const void *bias, int64_t n, uint32_t &umax) {
    uint2 bw = make_uint2(0u, 0u);
    if (bias) bw = *reinterpret_cast<const uint2 *>(static_cast<const uint16_t *>(bias) + n);
    return make_uint2(finish_pair<OUT_BF16>(v[0], v[1], bias != nullptr, bw.x, umax), finish_pair<OUT_BF16>(v[2], v[3], bias != nullptr, bw.y, umax));
}
template <bool OUT_BF16>
FOS_DEVICE uint32_t pack_outputs2(float v0, float v1, const void *bias, int64_t n, uint32_t &umax) {
    uint32_t bw = 0u;
    if (bias) bw = *reinterpret_cast<const uint32_t *>(static_cast<const uint16_t *>(bias) + n);
    return finish_pair<OUT_BF16>(v0, v1, bias != nullptr, bw, umax);
}

// max|D| for the caller that quantizes D next: the halves of `umax` hold the magnitude bits of the largest
// values this lane stored, as finish_pair folds them (0 for a lane that stored nothing).  At most one vector atomic per
// workgroup on the unsigned image of the value (non-negative floats order like their bits, NaN above all);
// every lane of the WAVES wavefronts must call it.  `words`: WAVES words of LDS nobody else uses any more.
//
// The atomics of a launch all go to one address and are served one after the other, about 12 ns each:
// bound by that chain, not by the reduction.  Workgroups of one generation end together, so that almost
// all of them find a smaller maximum in the word: with one atomic per wavefront a 2048 x 4096 x 4096 product
// took 75 us against 64 without the maximum (1024 wavefronts), and the reduction of a 128 x 4096 output's two partials
// 25 us (2048).  One per workgroup after a maximum in LDS: whole linear layers, quantization of the activation
// included, 128 x 14336 -> 4096 53.6 -> 39.9 us and 2048 x 4096 -> 4096 79.4 -> 76.2 us.
template <bool OUT_BF16, int WAVES>
FOS_DEVICE void fold_amax(float *d_amax, uint32_t umax, uint32_t *words) {
    const uint32_t top = (umax & 0xffffu) > (umax >> 16) ? umax & 0xffffu : umax >> 16;
    uint32_t r = top > (OUT_BF16 ? 0x7f80u : 0x7c00u) ? 0x7fc00000u : f2u(widen_out<OUT_BF16>(top));
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const uint32_t other = (uint32_t)__shfl_xor((int)r, off);
        r = other > r ? other : r;
    }
    if constexpr (WAVES > 1) {
        if ((threadIdx.x & 63) == 0) words[threadIdx.x >> 6] = r;
        __syncthreads();
        if (threadIdx.x < 64) {
#pragma unroll
            for (int w = 0; w < WAVES; ++w) r = words[w] > r ? words[w] : r;
        }
    }
    // (a workgroup first looks whether its value would change anything: a late one's seldom does)
    if (threadIdx.x == 0) {
        unsigned int *word = reinterpret_cast<unsigned int *>(d_amax);
        if (r > __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(word, r);
    }
}

// The two E4M3 bytes in the low 16 bits of `w` -> fp16 pair {s0, s1} (one hardware
// convert; exact, sub-normals included -- checked against the OCP decode of all 256 bytes).
FOS_DEVICE half2_t e4m3x2_to_half2(uint32_t w) {
    return __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, false);
}

// 8 packed codes (one 32-bit word) times a block scale -> 8 fp16 in k order.
FOS_DEVICE half8_t dequant8(uint32_t word, half2_t s) {
    half2_t p0 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(word, 1.0f, 0) * s;
    half2_t p1 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(word, 1.0f, 1) * s;
    half2_t p2 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(word, 1.0f, 2) * s;
    half2_t p3 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(word, 1.0f, 3) * s;
    half8_t r = {p0.x, p0.y, p1.x, p1.y, p2.x, p2.y, p3.x, p3.y};
    return r;
}

// 8 packed IF4 codes times their block scale -> 8 fp16 in k order.  A block holds E2M1 codes or (`integer`) two's
// complement integers q with the value RN16(6/7 q), and the product with the scale is rounded to fp16: the
// numbers the dequantization of the format is defined by (src/fouroversix/quantize/backend.py:89-160).
// Blocks differ from lane to lane, so both decodings are formed and one is selected: 34 instructions a word
// against 8 for E2M1 alone, and what bounds a product that converts inside its loop (layer of 2048 x 4096 -> 4096 110 us, with both
// operands converted ahead 80; two dequantize kernels, a library fp32 product and the conversion of its result took
// 570).  Integers: q + 8 = nibble ^ 8 is a byte 0 .. 15, which E4M3 reads as (q + 8) / 512 (the
// sub-normals run on into the first normal binade); 6/7 q is then formed from a two-part constant, equal to the rounded
// product for all 16 integers.
FOS_DEVICE void if4_integer_bytes(uint32_t word, uint32_t (&pairs)[2]) {
    const uint32_t u = word ^ 0x88888888u, even = u & 0x0f0f0f0fu, odd = (u >> 4) & 0x0f0f0f0fu;
    pairs[0] = __builtin_amdgcn_perm(odd, even, 0x05010400u);
    pairs[1] = __builtin_amdgcn_perm(odd, even, 0x07030602u);
}
FOS_DEVICE half2_t if4_sevenths(half2_t x) {
    constexpr _Float16 hi = (_Float16)(6.0 / 7.0), lo = (_Float16)(6.0 / 7.0 - (double)hi);
    const half2_t k512 = {(_Float16)512.0f, (_Float16)512.0f}, m8 = {(_Float16)-8.0f, (_Float16)-8.0f}, hi2 = {hi, hi}, lo2 = {lo, lo};
    const half2_t q = __builtin_elementwise_fma(x, k512, m8);
    return __builtin_elementwise_fma(q, hi2, q * lo2);
}
FOS_DEVICE half8_t dequant8_if4(uint32_t word, half2_t s, bool integer) {
    uint32_t pairs[2];
    if4_integer_bytes(word, pairs);
    auto sevenths = [](half2_t x) { return if4_sevenths(x); };
    auto pick = [&](half2_t i, half2_t f) {
        return __builtin_bit_cast(half2_t, integer ? __builtin_bit_cast(uint32_t, i) : __builtin_bit_cast(uint32_t, f)) * s;
    };
    const half2_t p0 = pick(sevenths(__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(pairs[0], 1.0f, false)),
                            __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(word, 1.0f, 0));
    const half2_t p1 = pick(sevenths(__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(pairs[0], 1.0f, true)),
                            __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(word, 1.0f, 1));
    const half2_t p2 = pick(sevenths(__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(pairs[1], 1.0f, false)),
                            __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(word, 1.0f, 2));
    const half2_t p3 = pick(sevenths(__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(pairs[1], 1.0f, true)),
                            __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(word, 1.0f, 3));
    half8_t r = {p0.x, p0.y, p1.x, p1.y, p2.x, p2.y, p3.x, p3.y};
    return r;
}

// One word of block `blk` (0, 1) of the two whose scale bytes are the low 16 bits of `two`.
template <bool IF4>
FOS_DEVICE half8_t dequant_word(uint32_t word, uint32_t two, int blk) {
    const half2_t s2 = e4m3x2_to_half2(IF4 ? two & 0x7f7fu : two);
    const half2_t s = blk ? __builtin_shufflevector(s2, s2, 1, 1) : __builtin_shufflevector(s2, s2, 0, 0);
    if constexpr (IF4) return dequant8_if4(word, s, (two & (blk ? 0x8000u : 0x80u)) != 0);
    else return dequant8(word, s);
}

// Output types of the tile kernels; kOutPartial: FP32 partial sums of a split of K.
enum { kOutF16 = 0, kOutBF16 = 1, kOutPartial = 2 };

}  // namespace fos
