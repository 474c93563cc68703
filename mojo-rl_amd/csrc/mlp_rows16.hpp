// Pieces of the kernels that take a net's rows in tiles of 16 or 32 on the 16-row matrix instructions (the fused update,
// mrl_fb.hip; the layer API, mrl_rows.hip; the policy step, mrl_policy.hip).
#pragma once
#include "mrl_device.hpp"
#include "mlp_tile.hpp"
#include "mlp_tile16.hpp"
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

constexpr int rows_threads(int H) { return H == 64 ? 256 : 512; }

// a row's run of 4 NT consecutive floats, 16 bytes at a time where the address allows it
template <int N>
MRL_DEV void store_run(float *p, const float (&y)[N], bool vec) {
    if (vec) {
#pragma unroll
        for (int j = 0; j < N; j += 4) *reinterpret_cast<f32x4 *>(p + j) = f32x4{y[j], y[j + 1], y[j + 2], y[j + 3]};
    } else {
#pragma unroll
        for (int j = 0; j < N; ++j) p[j] = y[j];
    }
}

// Forward of 16 rows by a workgroup of T threads.  Both hidden layers are computed transposed (output columns on the
// accumulator's rows), so that a lane ends up with 4 NT consecutive columns of one batch row, which it writes to LDS and to
// the cache in wide pieces.  k ascends through every product, so the bits are those of the 32-row tile (mlp_tile16.hpp).
// The hooks see what a caller keeps: on_x(row, input, value), on_layer0 / on_layer1(row, first column, RUN columns before and
// after the activation).  The head's outputs are in l.ys [16][PA_MAX + 1], behind a barrier, at the end.
template <int H, int ACT>
struct Rows16Forward {
    static constexpr int T = rows_threads(H), NW = T / 64, NT = H / 16 / NW, R = PR16, RUN = 4 * NT;
    static constexpr int FLD = H + 20, K0 = PIN_MAX / 4, KS = H / 4;
    static_assert(NT == 1 || NT == 2, "one float or one float2 of a weight row per lane");
    struct Lds {
        __align__(16) float h1f[R * FLD];
        __align__(16) float w2s[HEAD_LDS(H)];
        float xs[R * XS_LD];
        float h2[R * (H + 1)];
        float ys[R * (PA_MAX + 1)];
    };
    template <class OnX, class OnLayer0, class OnLayer1>
    static MRL_DEV void run(Lds &l, const float *__restrict__ params, const float *__restrict__ x, int nrow, int IN, int A,
                            bool GAUSS, OnX &&on_x, OnLayer0 &&on_layer0, OnLayer1 &&on_layer1) {
        const int t = threadIdx.x, lane = t & 63, w = t >> 6, g = lane >> 4, n = lane & 15;
        const int col_w = 16 * NT * w + NT * n;        // this lane's weight columns; tile q holds column col_w + q
        const int col_d = 16 * NT * w + RUN * g;       // its output columns, RUN of them, of batch row n
        const float *W0 = params, *b0 = params + IN * H, *W1 = b0 + H, *b1 = W1 + H * H;

        // ---- Everything from global memory is requested first, the rows ahead of the weights that hide behind them.  A lane
        // past the last row or input asks for the last one's value and drops it when it is used: behind a branch of its own,
        // or with the head's copy into LDS in between, a request would wait for the ones before it.
        constexpr int XQ = (R * 16 + T - 1) / T;
        float xa[XQ], xb[XQ];
#pragma unroll
        for (int q = 0; q < XQ; ++q) {
            const float *xr = x + min((t + q * T) >> 4, nrow - 1) * IN;
            const int j = t & 15;
            xa[q] = xr[min(j, IN - 1)];
            xb[q] = xr[min(j + 16, IN - 1)];
        }
        float w0[K0][NT], bias0[RUN], bias1[RUN];
#pragma unroll
        for (int s = 0; s < K0; ++s)
            if (s == 0 || 4 * s < IN) {
#pragma unroll
                for (int q = 0; q < NT; ++q) w0[s][q] = W0[min(4 * s + g, IN - 1) * H + col_w + q];
            }
#pragma unroll
        for (int j = 0; j < RUN; ++j) { bias0[j] = b0[col_d + j]; bias1[j] = b1[col_d + j]; }
        HeadLoads<H, T> head;
        head.load(params + IN * H + H + H * H + H, A, GAUSS, t);
        __builtin_amdgcn_sched_barrier(0);
        float w1[KS][NT];
#pragma unroll
        for (int s = 0; s < KS; ++s)
#pragma unroll
            for (int q = 0; q < NT; ++q) w1[s][q] = W1[(4 * s + g) * H + col_w + q];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < XQ; ++q) {
            const int r = (t + q * T) >> 4, j = t & 15;
            if (r < R) {
                if (j < IN) l.xs[r * XS_LD + j] = r < nrow ? xa[q] : 0.0f;
                if (j + 16 < IN) l.xs[r * XS_LD + j + 16] = r < nrow ? xb[q] : 0.0f;
                if (r < nrow) {
                    if (j < IN) on_x(r, j, xa[q]);
                    if (j + 16 < IN) on_x(r, j + 16, xb[q]);
                }
            }
        }
        head.store(l.w2s, A, GAUSS, t);
        __syncthreads();

        // ---- layer 0: D[column 4 g + v of tile q][batch row n]
        {
            f32x4 d[NT];
#pragma unroll
            for (int q = 0; q < NT; ++q) d[q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s = 0; s < K0; ++s) {
                if (4 * s < IN) {
                    const float xk = 4 * s + g < IN ? l.xs[n * XS_LD + 4 * s + g] : 0.0f;
#pragma unroll
                    for (int q = 0; q < NT; ++q) d[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(4 * s + g < IN ? w0[s][q] : 0.0f, xk, d[q], 0, 0, 0);
                }
            }
            float pre[RUN], y[RUN];
#pragma unroll
            for (int j = 0; j < RUN; ++j) {
                pre[j] = d[j % NT][j / NT] + bias0[j];
                y[j] = activate<ACT>(pre[j]);
            }
            store_run<RUN>(l.h1f + n * FLD + col_d, y, true);
            if (n < nrow) on_layer0(n, col_d, pre, y);
        }
        __syncthreads();

        // ---- layer 1
        {
            f32x4 d[NT];
#pragma unroll
            for (int q = 0; q < NT; ++q) d[q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                const float x = l.h1f[n * FLD + 4 * s + g];
#pragma unroll
                for (int q = 0; q < NT; ++q) d[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(w1[s][q], x, d[q], 0, 0, 0);
            }
            float pre[RUN], y[RUN];
#pragma unroll
            for (int j = 0; j < RUN; ++j) {
                pre[j] = d[j % NT][j / NT] + bias1[j];
                y[j] = activate<ACT>(pre[j]);
                l.h2[n * (H + 1) + col_d + j] = y[j];
            }
            if (n < nrow) on_layer1(n, col_d, pre, y);
        }
        __syncthreads();
        head16<H>(l.w2s, A, l.h2, l.ys, PA_MAX + 1, t, T);
        __syncthreads();
    }
};

}  // namespace mrl
