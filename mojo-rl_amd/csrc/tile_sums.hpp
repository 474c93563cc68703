// Where the pieces of a gradient lie that the row tiles and the weight-gradient launch leave, and how they are added up:
// shared by the sum kernel (mrl_mlp3.hip) and the kernel that goes on to Adam (mrl_update.hip).
#pragma once
#include <type_traits>
#include "mrl_device.hpp"
#include "mlp_tile.hpp"
#include "mlp_split.hpp"

namespace mrl {

// sum over a wavefront, the same in every lane: rows of sixteen by rotations, then the four rows (a twelfth of the time of
// six exchanges through the LDS crossbar)
MRL_DEV float dpp_wave_sum(float x) {
    x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x128, 0xf, 0xf, false));   // row_ror:8
    x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x124, 0xf, 0xf, false));   // row_ror:4
    x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x122, 0xf, 0xf, false));   // row_ror:2
    x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x121, 0xf, 0xf, false));   // row_ror:1
    auto row = [&](int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l)); };
    return (row(0) + row(16)) + (row(32) + row(48));
}

// Where the terms of a net's gradient are, element by element of the flat vector [W0; b0; W1; b1; W2; b2; log_std]: the H x H
// block in the batch splits' partial vectors or in the row tiles' pieces, the other weights in the tiles' pieces, bias rows
// and the log_std tail (Gaussian head) in the column sums that the tiles left.
struct SumNet {
    float *grads;
    const float *hidden, *thin, *db, *ls;
    int P, A;
    int hidden_stride, hidden_n;   // of the terms of the H x H block
    int thin_stride;               // floats per row tile in `thin`
};
struct SumNets {
    SumNet net[2];
    int n, IN, H, tiles;
    const int32_t *skip;   // as FwdLoss::skip, never null
};

// the n terms of an element: p, p + stride, ...
struct SumTerms { const float *p; int stride, n; };

// element e of the H x H block
MRL_DEV SumTerms hidden_terms(const SumNet &net, int e) { return {net.hidden + e, net.hidden_stride, net.hidden_n}; }

// Element i outside the H x H block.  (Selects: a branch per kind of element would fetch its own arguments one after the
// other, a few hundred cycles each.)
MRL_DEV SumTerms thin_terms(const SumNet &net, int IN, int H, int tiles, int i) {
    const int A = net.A, o1 = (IN + 1) * H, o2 = o1 + (H + 1) * H, o3 = o2 + (H + 1) * A;
    int at = i < o1 ? i : IN * H + i - o2, stride = net.thin_stride;
    const float *p = net.thin;
    const bool b0 = i >= IN * H && i < o1, b1 = i >= o1 && i < o2, b2 = i >= o2 + H * A, tail = i >= o3;
    at = b0 ? i - IN * H : b1 ? H + i - (o1 + H * H) : tail ? i - o3 : b2 ? 2 * H + i - (o2 + H * A) : at;
    stride = tail ? A : b0 || b1 || b2 ? 2 * H + PA_MAX : stride;
    p = tail ? net.ls : b0 || b1 || b2 ? net.db : p;
    return {p + at, stride, tiles};
}

typedef float f32x4a4 __attribute__((ext_vector_type(4), aligned(4)));

// The sum of a few terms V (float, or four neighbouring floats).  The chain of memory round trips is what this takes, so up
// to 64 registers of terms are requested at a time, and the last few of a number that is no multiple of 8 go out together as
// well: with a request at a time behind the last 16, the sum over 63 tiles took 8.7 us of a minibatch's 31 (H = 128, 1000
// rows), so 5.3.  They are added one after the other, or (TREE) what is requested together as a tree of neighbours, in the
// order it comes back.  The pieces of 16-row tiles take the tree: they are twice as many as those of 32-row tiles, and one
// after the other their roundings had made the gradients of 2048-row minibatches (H = 256, 24 inputs) less exact,
// 1.43e-7 -> 1.55e-7 off Float64; as a tree 0.75e-7, in the same time.
template <bool TREE, class V>
MRL_DEV V sum_terms(const SumTerms &terms) {
    const float *__restrict__ p = terms.p;
    const size_t stride = (size_t)terms.stride;
    int n = terms.n;
    typedef std::conditional_t<sizeof(V) == 4, float, f32x4a4> Load;
    constexpr int MOST = 256 / sizeof(V);
    V s = V{};
    auto whole = [&](auto width) {
        constexpr int W = decltype(width)::value;
        if constexpr (W <= MOST) {
            V v[W];
#pragma unroll
            for (int k = 0; k < W; ++k) v[k] = *reinterpret_cast<const Load *>(p + (size_t)k * stride);
            if constexpr (TREE) {
#pragma unroll
                for (int d = 1; d < W; d *= 2)
#pragma unroll
                    for (int k = 0; k < W; k += 2 * d) v[k] += v[k + d];
                s += v[0];
            } else {
#pragma unroll
                for (int k = 0; k < W; ++k) s += v[k];
            }
            p += W * stride;
            n -= W;
        }
    };
    while (n >= MOST) whole(std::integral_constant<int, MOST>{});
    if (MOST > 32 && n >= 32) whole(std::integral_constant<int, 32>{});
    if (MOST > 16 && n >= 16) whole(std::integral_constant<int, 16>{});
    if (n >= 8) whole(std::integral_constant<int, 8>{});
    if (n > 0) {
        V v[7];
#pragma unroll
        for (int k = 0; k < 7; ++k) {
            v[k] = *reinterpret_cast<const Load *>(p);
            p += k + 1 < n ? stride : 0;   // (past the end: the last term again, not added)
        }
#pragma unroll
        for (int k = 0; k < 7; ++k) s += k < n ? v[k] : V{};
    }
    return s;
}

}  // namespace mrl
