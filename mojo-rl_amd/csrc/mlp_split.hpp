// fp32 products on the bf16 matrix cores.
//
// A float of at least 2^-110 is the exact sum of three bf16 values (8 + 8 + 8 significant bits, each the rounding of what
// the ones before it left), so a product of two floats is nine bf16 products, each exact in fp32.  The six largest are kept:
//   a b  =  a1 b1 + (a1 b2 + a2 b1) + (a1 b3 + a2 b2 + a3 b1),
// what is left out is at most 2^-24 |a b| (a and b just above a power of two) and 2^-27.5 |a b| in the root mean square,
// where rounding one fp32 product costs up to 2^-24 and 2^-25.2.  The sums run in the
// matrix cores' fp32 accumulators, the five small products in one of their own, so that a sum over K terms is rounded
// K / 32 times at its full size where a chain of fp32 multiply-adds is rounded K times: against Float64 the results are
// closer than those of v_mfma_f32_* (tests/test_gpu_split.py).  v_mfma_f32_16x16x32_bf16 does in 16 cycles what eight
// v_mfma_f32_16x16x4_f32 do in 256; with six of them per product this is 2.7 times the fp32 rate.
//
// The ends of the range (tests/test_gpu_split_range.py).  bf16's subnormals go through the matrix cores as they are, in
// steps of 2^-133: a value below 2^-110 is off by up to 2^-134, which the fp32 instructions would keep.  A finite value
// that rounds past bf16's largest takes that as its first piece.  An infinity has the pieces (inf, NaN, NaN): the
// first products alone tell what fp32 gives, and where they add up to an infinity the small ones are not added
// (split_sum).  Products and sums overflow where fp32's do, within the 2^-8 that the first pieces differ from their value.
//
// Operand layout of v_mfma_f32_16x16x32_bf16, lane = 16 g + n:  A[row n][k = 8 g + j], B[k = 8 g + j][column n],
// j = 0 .. 7 (16 bytes per lane)  ->  D[row 4 g + v][column n], v = 0 .. 3.
#pragma once
#include "mrl_device.hpp"

namespace mrl {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x8 __attribute__((ext_vector_type(8)));

constexpr int SPLIT = 3;   // pieces per float

constexpr float SPLIT_TOP = 0x1.fep127f, SPLIT_OVER = 0x1.ffp127f;   // bf16's largest value; from here on a float rounds past it

template <int N, class F, class B>
MRL_DEV void split_n(const F x, B (&p)[SPLIT]) {
    F r = x;
    float top = 0.0f;
#pragma unroll
    for (int j = 0; j < N; ++j) top = fmaxf(top, fabsf(x[j]));
    p[0] = __builtin_convertvector(r, B);
    if (top >= SPLIT_OVER) {   // (hardly ever: a branch costs less than N selects)
#pragma unroll
        for (int j = 0; j < N; ++j)
            if (fabsf(x[j]) >= SPLIT_OVER && fabsf(x[j]) < INFINITY) p[0][j] = (__bf16)copysignf(SPLIT_TOP, x[j]);
    }
#pragma unroll
    for (int i = 1; i < SPLIT; ++i) {
        r = r - __builtin_convertvector(p[i - 1], F);
        p[i] = __builtin_convertvector(r, B);
    }
}
MRL_DEV void split4(const f32x4 x, bf16x4 (&p)[SPLIT]) { split_n<4>(x, p); }
MRL_DEV void split8(const f32x8 x, bf16x8 (&p)[SPLIT]) { split_n<8>(x, p); }

// hi += a1 b1, lo += the five smaller products of one k-step of 32
MRL_DEV void mfma_split(const bf16x8 (&a)[SPLIT], const bf16x8 (&b)[SPLIT], f32x4 &hi, f32x4 &lo) {
    lo = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[2], b[0], lo, 0, 0, 0);
    hi = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], b[0], hi, 0, 0, 0);
    lo = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[1], b[1], lo, 0, 0, 0);
    lo = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], b[2], lo, 0, 0, 0);
    lo = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[1], b[0], lo, 0, 0, 0);
    lo = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], b[1], lo, 0, 0, 0);
}

// what hi and lo add up to; a lo that is NaN, beside an infinite (or NaN) hi, becomes a finite number (v_med3_f32 takes the
// lowest of the others), which leaves hi what it is
MRL_DEV float split_sum(float hi, float lo) { return hi + __builtin_amdgcn_fmed3f(lo, -__FLT_MAX__, __FLT_MAX__); }

// A hidden layer's weights W [H, H] as operands, split, in the order the lanes read them: piece p of the 8 elements
// that lane `lane` holds in k-step ks (32 of the contracted index) of column tile ct (16 of the other index) starts at
// element split_frag<H>(ks, ct, p, lane).  Forward: contracted = row of W; backward (W^T): contracted = column of W.
template <int H>
MRL_DEV size_t split_frag(int ks, int ct, int p, int lane) {
    return ((((size_t)ks * (H / 16) + ct) * SPLIT + p) * 64 + lane) * 8;
}
constexpr size_t split_elems(int H) { return (size_t)SPLIT * H * H; }   // bf16 elements of one orientation

}  // namespace mrl
