// Pieces of the kernels that take a net's rows in tiles of 16 or 32 on the 16-row matrix instructions (the fused update,
// mrl_fb.hip; the layer API, mrl_rows.hip).
#pragma once
#include "mrl_device.hpp"
#include "mlp_tile.hpp"
#include "mlp_split.hpp"

namespace mrl {

template <int ACT>
MRL_DEV float act_deriv_out(float y) {
    if (ACT == 1) return y > 0.0f ? 1.0f : 0.0f;
    if (ACT == 2) return 1.0f - y * y;
    return 1.0f;
}

// sum over the sixteen lanes of a row (DPP rotations within the row), on all of them
MRL_DEV float row16_sum(float x) {
    x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x128, 0xf, 0xf, false));   // row_ror:8
    x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x124, 0xf, 0xf, false));   // row_ror:4
    x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x122, 0xf, 0xf, false));   // row_ror:2
    x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x121, 0xf, 0xf, false));   // row_ror:1
    return x;
}

// A tile's rows of column tile ct (RT = 1: of ct and ct + 1) of f [16 RT][LD] (LDS), split, as the operand pieces that a
// product contracted over the batch rows reads (k-step = 32 rows): lane 16 g + n holds rows 8 g .. 8 g + 7 of column n.
// A tile of 16 rows fills half a k-step: it takes two column tiles per wavefront; the last tile of an odd count puts
// zeros where the other half would be.
template <int H, int RT, int LD>
MRL_DEV void batch_operand(const float *f, unsigned short *dst, int ct, int lane) {
    const int g = lane >> 4, n = lane & 15;
    const int c = ct + (RT == 1 ? g >> 1 : 0), rg = RT == 1 ? g & 1 : g;
    const int ks = RT == 1 ? blockIdx.x >> 1 : blockIdx.x, gs = RT == 1 ? 2 * (blockIdx.x & 1) + rg : g;
    f32x8 x;
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = f[(8 * rg + j) * LD + 16 * c + n];
    bf16x8 p[SPLIT];
    split8(x, p);
    const bool pad = RT == 1 && blockIdx.x == gridDim.x - 1 && (blockIdx.x & 1) == 0;
#pragma unroll
    for (int i = 0; i < SPLIT; ++i) {
        *reinterpret_cast<bf16x8 *>(dst + split_frag<H>(ks, c, i, 16 * gs + n)) = p[i];
        if (pad) *reinterpret_cast<uint4 *>(dst + split_frag<H>(ks, c, i, 16 * (gs + 2) + n)) = make_uint4(0, 0, 0, 0);
    }
}

constexpr int fb_threads(int H) { return H == 64 ? 256 : 512; }

}  // namespace mrl
