// The layer API's passes over the agents' three-layer nets  IN -> H -> H -> out  (H in {64, 128, 256}, IN <= 32, out <= 8
// or a StochasticActor head of <= 8): forward with the reference's per-layer cache, and backward from the caller's output
// gradient to the parameter gradients and, if asked for, the gradient of the input (deep_rl/model/sequential.mojo:
// 104-133, 867-953; linear{,_relu,_tanh}.mojo, stochastic_actor.mojo).  A workgroup takes 16 (backward: or 32) batch rows
// through all three layers.  Products that reach a caller's output directly run on v_mfma_f32_16x16x4_f32.
//
// What bounds both: the chain of phases of one tile, of which the H x H product's fp32 matrix time is half (H = 256: 64
// k-steps of 32 cycles on each of a wavefront's column tiles, two wavefronts per SIMD); the weights a wavefront multiplies
// are requested before anything else needs them, whole, into registers.  us, 24 inputs, tanh, 8 outputs, against a 32-row
// forward and a backward that ran layer by layer as soon as the input gradient was asked for (9 launches):
//   forward with cache   H = 64, 33 rows 11.4 -> 5.7;  H = 128, 1000 rows 42.0 -> 7.3;  H = 256, 4096 rows 22.6 -> 17.3
//   backward, grad_in    H = 64, 33 rows 40.9 -> 8.8;  H = 128, 1000 rows 89.3 -> 18.8;  H = 256, 4096 rows 154 -> 38
//   backward, no grad_in H = 64, 33 rows 20.9 -> 8.7;  H = 128, 1000 rows 76.6 -> 16.8;  H = 256, 4096 rows 48.9 -> 35.2
#include "mrl_host.hpp"
#include "mrl_device.hpp"
#include "mlp_tile.hpp"
#include "mlp_tile16.hpp"
#include "mlp_rows16.hpp"
#include "mlp3.hpp"

namespace mrl {

// Forward with the reference's per-layer cache (null: none), Rows16Forward per workgroup.
template <int H, int ACT>
__global__ __launch_bounds__(rows_threads(H)) void mlp3_fwd16_kernel(int B, int IN, Mlp3Net nn) {
    using F = Rows16Forward<H, ACT>;
    constexpr int T = F::T, RUN = F::RUN, R = PR16;
    __shared__ typename F::Lds lds;
    float *__restrict__ cache = nn.cache;
    const int A = nn.A;
    const bool GAUSS = nn.gauss != 0;
    const int t = threadIdx.x;
    const long row0 = (long)blockIdx.x * R;
    const int nrow = (int)min((long)R, B - row0);
    float *c0 = cache, *c1 = cache + (size_t)B * (IN + H), *c2 = c1 + (size_t)B * 2 * H;
    const bool vec0 = IN % 4 == 0 && (reinterpret_cast<uintptr_t>(c0) & 15) == 0;
    const bool vec1 = (reinterpret_cast<uintptr_t>(c1) & 15) == 0;   // (c2 lies a multiple of 2 H floats behind it)
    F::run(lds, nn.params, nn.x + row0 * IN, nrow, IN, A, GAUSS,
           [&](int r, int j, float v) {
               if (cache != nullptr) c0[(row0 + r) * (IN + H) + j] = v;
           },
           [&](int n, int col, const float (&pre)[RUN], const float (&y)[RUN]) {
               if (cache == nullptr) return;
               store_run<RUN>(c0 + (row0 + n) * (IN + H) + IN + col, ACT == 1 ? pre : y, vec0);
               store_run<RUN>(c1 + (row0 + n) * (2 * H) + col, y, vec1);
           },
           [&](int n, int col, const float (&pre)[RUN], const float (&y)[RUN]) {
               if (cache == nullptr) return;
               store_run<RUN>(c1 + (row0 + n) * (2 * H) + H + col, ACT == 1 ? pre : y, vec1);
               store_run<RUN>(c2 + (row0 + n) * H + col, y, vec1);
           });
    const int ld = GAUSS ? 2 * A : A;
    for (int i = t; i < nrow * ld; i += T) {
        const int r = i / ld, a = i - r * ld;
        float v;
        if (a < A) {
            v = lds.ys[r * (PA_MAX + 1) + a];
        } else {   // state-independent log_std, clamped (deep_rl/model/stochastic_actor.mojo:260-275)
            v = lds.w2s[HEAD_LOG_STD(H) + (a - A)];
            v = v < -5.0f ? -5.0f : (v > 2.0f ? 2.0f : v);
        }
        nn.out[(row0 + r) * ld + a] = v;
    }
}

// Backward of 16 RT rows: grad_out [B, ld] (ld = A, or 2 A for the Gaussian head: mean gradients first) goes back through
// head, layer 1 and layer 0, the activations come from the cache.  Leaves per tile the bias and thin-layer gradients and
// the log_std column sums; the hidden layer's weight gradient as one more piece (dw_in_tiles) or h1 and g1 split, as
// operands of dw_frag_kernel; and grad_in [B, IN] itself (null: not wanted).
// The two thin products beside it (dW0 = x^T g0, grad_in = g0 W0^T) are contracted over rows and over columns: g0 is the
// first one's operand where the accumulator leaves it, and goes through LDS for the second, each wavefront its own columns.
template <int H, int ACT, int RT>
__global__ __launch_bounds__(rows_threads(H)) void mlp3_bwd_kernel(int B, int IN, Mlp3Net nn, int dw_in_tiles) {
    constexpr int T = rows_threads(H), NW = T / 64, NT = H / 16 / NW, R = 16 * RT, NS = H / 16;
    constexpr int XLD = PIN_MAX + 1, FLD = H + 20, GLD = 2 * PA_MAX + 1, ILD = PIN_MAX + 1;
    constexpr int HQ = (R * H / 4 + T - 1) / T;
    constexpr bool DW_IN_TILE = H <= 128, BATCH_OPERANDS = H > 64 && NT % (2 / RT) == 0;
    constexpr bool G0_ON_H1 = !DW_IN_TILE;     // (nobody else reads a wavefront's columns of h1 any more)
    __shared__ float xs[R * XLD];
    __shared__ __align__(16) float h1f[R * FLD];
    __shared__ __align__(16) float h2f[R * FLD];
    __shared__ __align__(16) float g0s[G0_ON_H1 ? 4 : R * FLD];
    // (g1 lies over h2: a wavefront writes only columns whose h2 it alone reads, after it has read them)
    float *g1f = h2f, *g0f = G0_ON_H1 ? h1f : g0s;
    __shared__ __align__(16) float w2s[HEAD_LDS(H)];
    __shared__ float g2s[R * GLD];
    __shared__ float red[NW * R * ILD];
    const float *__restrict__ params = nn.params, *__restrict__ cache = nn.cache, *__restrict__ grad_out = nn.grad_out;
    const int A = nn.A;
    const bool GAUSS = nn.gauss != 0;
    const int ld = GAUSS ? 2 * A : A;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, g = lane >> 4, n = lane & 15;
    const long row0 = (long)blockIdx.x * R;
    const int nrow = (int)min((long)R, B - row0);
    const float *c0 = cache, *c1 = cache + (size_t)B * (IN + H), *c2 = c1 + (size_t)B * 2 * H;
    const float *W0 = params, *W1 = params + IN * H + H;
    float *__restrict__ db_part = nn.db_part + (size_t)blockIdx.x * (2 * H + PA_MAX);
    float *__restrict__ thin_part = nn.thin_part + (size_t)blockIdx.x * (size_t)nn.thin_stride;

    // ---- everything from global memory is requested first, the rows ahead of the weights that hide behind them (as in
    // Rows16Forward: a lane past the end asks for the last value and drops it when it is used)
    f32x4 v1[HQ], v2[HQ];
    const bool vec = (reinterpret_cast<uintptr_t>(c1) & 15) == 0;    // (c2 lies a multiple of 2 H floats behind it)
#pragma unroll
    for (int q = 0; q < HQ; ++q) {
        const int e = 4 * (t + q * T), r = min(e / H, nrow - 1), c = e % H;
        const float *s1 = c1 + (row0 + r) * (2 * H) + c, *s2 = c2 + (row0 + r) * H + c;
        if (vec) {
            v1[q] = *reinterpret_cast<const f32x4 *>(s1);
            v2[q] = *reinterpret_cast<const f32x4 *>(s2);
        } else {
            v1[q] = f32x4{s1[0], s1[1], s1[2], s1[3]};
            v2[q] = f32x4{s2[0], s2[1], s2[2], s2[3]};
        }
    }
    constexpr int XQ = (R * 16 + T - 1) / T, GQ = (R * GLD + T - 1) / T;
    float xa[XQ], xb[XQ], gq[GQ];
#pragma unroll
    for (int q = 0; q < XQ; ++q) {
        const float *x = c0 + (row0 + min((t + q * T) >> 4, nrow - 1)) * (IN + H);
        const int j = t & 15;
        xa[q] = x[min(j, IN - 1)];
        xb[q] = x[min(j + 16, IN - 1)];
    }
#pragma unroll
    for (int q = 0; q < GQ; ++q) {
        const int i = t + q * T, r = i / GLD, a = i - r * GLD;
        gq[q] = grad_out[(row0 + min(r, nrow - 1)) * ld + min(a, ld - 1)];
    }
    HeadLoads<H, T> head;
    head.load(W1 + H * H + H, A, false, t);
    __builtin_amdgcn_sched_barrier(0);
    // W1^T as operand: k-slot g of step v in group s is column 16 s + 4 g + v of W1, for both operands
    f32x4 w1[NT][NS];
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int q = 0; q < NT; ++q)
            w1[q][s] = *reinterpret_cast<const f32x4 *>(W1 + (size_t)(16 * (NT * w + q) + n) * H + 16 * s + 4 * g);
    f32x4 w0[2][NT];
#pragma unroll
    for (int it = 0; it < 2; ++it)
#pragma unroll
        for (int q = 0; q < NT; ++q) {
            if (nn.grad_in != nullptr)
                w0[it][q] = *reinterpret_cast<const f32x4 *>(W0 + min(16 * it + n, IN - 1) * H + 16 * (NT * w + q) + 4 * g);
        }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < HQ; ++q) {
        const int e = 4 * (t + q * T), r = e / H, c = e % H;
        if (r < R) {
            const f32x4 none = {0.0f, 0.0f, 0.0f, 0.0f};
            *reinterpret_cast<f32x4 *>(h1f + r * FLD + c) = r < nrow ? v1[q] : none;
            *reinterpret_cast<f32x4 *>(h2f + r * FLD + c) = r < nrow ? v2[q] : none;
        }
    }
#pragma unroll
    for (int q = 0; q < XQ; ++q) {
        const int r = (t + q * T) >> 4, j = t & 15;
        if (r < R) {
            if (j < IN) xs[r * XLD + j] = r < nrow ? xa[q] : 0.0f;
            if (j + 16 < IN) xs[r * XLD + j + 16] = r < nrow ? xb[q] : 0.0f;
            if (j == 0) xs[r * XLD + IN] = 1.0f;     // the bias gradient of layer 0 as row IN of x^T g0
        }
    }
#pragma unroll
    for (int q = 0; q < GQ; ++q) {
        const int i = t + q * T, r = i / GLD, a = i - r * GLD;
        if (i < R * GLD) g2s[i] = r < nrow && a < ld ? gq[q] : 0.0f;
    }
    head.store(w2s, A, false, t);
    __syncthreads();

    // ---- back through the head and layer 1's activation: g1^T[column 4 g + v][batch row n]
    {
        float w2[NT][PA_MAX / 4], gb[RT][PA_MAX / 4], gr[4 * RT];
#pragma unroll
        for (int s = 0; s < PA_MAX / 4; ++s) {
#pragma unroll
            for (int q = 0; q < NT; ++q) w2[q][s] = w2s[(16 * (NT * w + q) + n) * PA_MAX + 4 * s + g];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) gb[rt][s] = 4 * s + g < A ? g2s[(16 * rt + n) * GLD + 4 * s + g] : 0.0f;
        }
#pragma unroll
        for (int s = 0; s < 4 * RT; ++s) gr[s] = g2s[(4 * s + g) * GLD + n];
        f32x4 d[NT][RT], d2[NT], h2v[RT][NT];
#pragma unroll
        for (int q = 0; q < NT; ++q) {
            d2[q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                d[q][rt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                h2v[rt][q] = *reinterpret_cast<const f32x4 *>(h2f + (16 * rt + n) * FLD + 16 * (NT * w + q) + 4 * g);
            }
        }
#pragma unroll
        for (int s = 0; s < PA_MAX / 4; ++s)
#pragma unroll
            for (int q = 0; q < NT; ++q)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt)
                    d[q][rt] = __builtin_amdgcn_mfma_f32_16x16x4f32(w2[q][s], gb[rt][s], d[q][rt], 0, 0, 0);
        // dW2[col][a] of the tile = sum over rows of h2[row][col] g2[row][a]
#pragma unroll
        for (int s = 0; s < 4 * RT; ++s)
#pragma unroll
            for (int q = 0; q < NT; ++q)
                d2[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(h2f[(4 * s + g) * FLD + 16 * (NT * w + q) + n], gr[s], d2[q], 0, 0, 0);
        __builtin_amdgcn_wave_barrier();   // (h2 of these columns has been read by every lane)
        asm volatile("" : : : "memory");
#pragma unroll
        for (int q = 0; q < NT; ++q) {
            const int c = 16 * (NT * w + q) + 4 * g;
            f32x4 cs = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                f32x4 y;
#pragma unroll
                for (int v = 0; v < 4; ++v) y[v] = d[q][rt][v] * act_deriv_out<ACT>(h2v[rt][q][v]);
                cs = cs + y;
                *reinterpret_cast<f32x4 *>(g1f + (16 * rt + n) * FLD + c) = y;
            }
            // bias gradient of layer 1: over the rows, which are the sixteen lanes n
#pragma unroll
            for (int v = 0; v < 4; ++v) cs[v] = row16_sum(cs[v]);
            if (n == 0) *reinterpret_cast<f32x4 *>(db_part + H + c) = cs;
            if (n < A) {
#pragma unroll
                for (int v = 0; v < 4; ++v) thin_part[(size_t)IN * H + (size_t)(c + v) * A + n] = d2[q][v];
            }
        }
        if (BATCH_OPERANDS && !dw_in_tiles) {
            // h1 and g1 out to the weight-gradient launch (g1's columns were written by this wavefront)
            asm volatile("" : : : "memory");
#pragma unroll
            for (int q = 0; q < NT; q += 2 / RT) {
                batch_operand<H, RT, FLD>(h1f, nn.h1q, NT * w + q, lane);
                batch_operand<H, RT, FLD>(g1f, nn.g1q, NT * w + q, lane);
            }
        }
    }
    if (w == NW - 1 && lane < ld) {   // column sums of the tile: bias gradient of the head, log_std gradient
        float s = 0.0f;
#pragma unroll
        for (int r = 0; r < R; ++r) s += g2s[r * GLD + lane];
        if (lane < A) db_part[2 * H + lane] = s;
        else nn.ls_part[(long)blockIdx.x * A + (lane - A)] = s;
    }
    __syncthreads();

    // ---- dh1 = g1 W1^T: D[batch row 4 g + v][column n]; two chains per tile
    {
        f32x4 acc[2][NT][RT];
#pragma unroll
        for (int q = 0; q < NT; ++q)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) acc[0][q][rt] = acc[1][q][rt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            f32x4 a[RT];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) a[rt] = *reinterpret_cast<const f32x4 *>(g1f + (16 * rt + n) * FLD + 16 * s + 4 * g);
#pragma unroll
            for (int v = 0; v < 4; ++v)
#pragma unroll
                for (int q = 0; q < NT; ++q)
#pragma unroll
                    for (int rt = 0; rt < RT; ++rt)
                        acc[v & 1][q][rt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[rt][v], w1[q][s][v], acc[v & 1][q][rt], 0, 0, 0);
        }
        float g0[NT][RT][4];
#pragma unroll
        for (int q = 0; q < NT; ++q)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    g0[q][rt][v] = (acc[0][q][rt][v] + acc[1][q][rt][v]) *
                                   act_deriv_out<ACT>(h1f[(16 * rt + 4 * g + v) * FLD + 16 * (NT * w + q) + n]);
        // dW0[i][c] of the tile = sum over rows of x[row][i] g0[row][c]; row IN of x^T holds ones
        for (int it = 0; 16 * it <= IN; ++it) {
            const int i = 16 * it + n;
            float x[RT][4];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int v = 0; v < 4; ++v) x[rt][v] = i <= IN ? xs[(16 * rt + 4 * g + v) * XLD + i] : 0.0f;
            f32x4 d[NT];
#pragma unroll
            for (int q = 0; q < NT; ++q) d[q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int v = 0; v < 4; ++v)
#pragma unroll
                    for (int q = 0; q < NT; ++q)
                        d[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[rt][v], g0[q][rt][v], d[q], 0, 0, 0);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int row = 16 * it + 4 * g + v;
                float *o = row < IN ? thin_part + (size_t)row * H : db_part;
                if (row <= IN) {
#pragma unroll
                    for (int q = 0; q < NT; ++q) o[16 * (NT * w + q) + n] = d[q][v];
                }
            }
        }
        if (nn.grad_in != nullptr) {
            // grad_in[r][i] = sum over c of g0[r][c] W0[i][c]: this wavefront's columns, the others' added below
            asm volatile("" : : : "memory");
#pragma unroll
            for (int q = 0; q < NT; ++q)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                    for (int v = 0; v < 4; ++v) g0f[(16 * rt + 4 * g + v) * FLD + 16 * (NT * w + q) + n] = g0[q][rt][v];
            __builtin_amdgcn_wave_barrier();
            asm volatile("" : : : "memory");
            f32x4 d[2][RT];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) d[0][rt] = d[1][rt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int q = 0; q < NT; ++q)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
                    const f32x4 a = *reinterpret_cast<const f32x4 *>(g0f + (16 * rt + n) * FLD + 16 * (NT * w + q) + 4 * g);
#pragma unroll
                    for (int v = 0; v < 4; ++v)
#pragma unroll
                        for (int it = 0; it < 2; ++it)
                            d[it][rt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[v], w0[it][q][v], d[it][rt], 0, 0, 0);
                }
#pragma unroll
            for (int it = 0; it < 2; ++it)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        red[(w * R + 16 * rt + 4 * g + v) * ILD + 16 * it + n] = d[it][rt][v];
        }
    }
    if constexpr (DW_IN_TILE) {
        // dW1[k][c] of the tile = sum over rows of h1[row][k] g1[row][c] as one more piece for the sum kernel
        if (dw_in_tiles) {
            float *o1 = thin_part + (size_t)IN * H + (size_t)H * A;
#pragma unroll
            for (int q = 0; q < NT; ++q) {
                const int c = 16 * (NT * w + q) + n;
                float b[4 * RT];
#pragma unroll
                for (int s = 0; s < 4 * RT; ++s) b[s] = g1f[(4 * s + g) * FLD + c];
#pragma unroll 4
                for (int kt = 0; kt < H / 16; ++kt) {
                    f32x4 d = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int s = 0; s < 4 * RT; ++s)
                        d = __builtin_amdgcn_mfma_f32_16x16x4f32(h1f[(4 * s + g) * FLD + 16 * kt + n], b[s], d, 0, 0, 0);
#pragma unroll
                    for (int v = 0; v < 4; ++v) o1[(size_t)(16 * kt + 4 * g + v) * H + c] = d[v];
                }
            }
        }
    }
    if (nn.grad_in == nullptr) return;
    __syncthreads();
    for (int e = t; e < nrow * IN; e += T) {
        const int r = e / IN, i = e - r * IN;
        float s = 0.0f;
#pragma unroll
        for (int k = 0; k < NW; ++k) s += red[(k * R + r) * ILD + i];
        nn.grad_in[row0 * IN + e] = s;
    }
}

template <int H>
static void launch_fwd16_h(mrl_ctx *ctx, int act, int batch, int IN, const Mlp3Net &nn) {
    const dim3 grid((batch + PR16 - 1) / PR16), block(rows_threads(H));
    if (act == 1) hipLaunchKernelGGL((mlp3_fwd16_kernel<H, 1>), grid, block, 0, ctx->stream, batch, IN, nn);
    else hipLaunchKernelGGL((mlp3_fwd16_kernel<H, 2>), grid, block, 0, ctx->stream, batch, IN, nn);
}
int launch_fwd16(mrl_ctx *ctx, int H, int act, int batch, int IN, const Mlp3Net &nn) {
    if (H == 256) launch_fwd16_h<256>(ctx, act, batch, IN, nn);
    else if (H == 128) launch_fwd16_h<128>(ctx, act, batch, IN, nn);
    else launch_fwd16_h<64>(ctx, act, batch, IN, nn);
    MRL_CHECK_LAUNCH();
    return MRL_OK;
}

template <int H, int ACT>
static void launch_bwd_h(mrl_ctx *ctx, int batch, int IN, int rows, const Mlp3Net &nn, int dw_in_tiles) {
    const dim3 grid((batch + rows - 1) / rows), block(rows_threads(H));
    if (rows == 16) hipLaunchKernelGGL((mlp3_bwd_kernel<H, ACT, 1>), grid, block, 0, ctx->stream, batch, IN, nn, dw_in_tiles);
    else hipLaunchKernelGGL((mlp3_bwd_kernel<H, ACT, 2>), grid, block, 0, ctx->stream, batch, IN, nn, dw_in_tiles);
}
int launch_bwd(mrl_ctx *ctx, int H, int act, int batch, int IN, int rows, const Mlp3Net &nn, bool dw_in_tiles) {
    if (H == 256 && act == 1) launch_bwd_h<256, 1>(ctx, batch, IN, rows, nn, dw_in_tiles);
    else if (H == 256) launch_bwd_h<256, 2>(ctx, batch, IN, rows, nn, dw_in_tiles);
    else if (H == 128 && act == 1) launch_bwd_h<128, 1>(ctx, batch, IN, rows, nn, dw_in_tiles);
    else if (H == 128) launch_bwd_h<128, 2>(ctx, batch, IN, rows, nn, dw_in_tiles);
    else if (act == 1) launch_bwd_h<64, 1>(ctx, batch, IN, rows, nn, dw_in_tiles);
    else launch_bwd_h<64, 2>(ctx, batch, IN, rows, nn, dw_in_tiles);
    MRL_CHECK_LAUNCH();
    return MRL_OK;
}

}  // namespace mrl
