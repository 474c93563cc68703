// Forward, PPO loss gradients and the way back of one row tile of a minibatch in one workgroup, for the agents'
// three-layer nets  IN -> H -> H -> out  (H in {64, 128, 256}, IN <= 32, out <= 8 or a StochasticActor head of <= 8).
//
// The minibatch never needs the activations outside the workgroup that made them: a tile of 16 RT rows is read from the
// rollout through the minibatch indices, goes forward, on to its loss gradients (deep_agents/ppo/ppo.mojo:285-378,
// 538-633; kernels.mojo:230-486) and its share of the KL test, and back through the three layers while h1 and h2 are in
// LDS.  What leaves the chip: outputs and head gradients, the tile's bias / thin-layer / (H <= 128) hidden-layer weight
// gradients, and for the H x H weight gradient of wide nets h1 and g1.  act' comes from the activation's output.
//
// The two H x H products per tile run on the bf16 matrix cores with split operands (mlp_split.hpp); the weights come
// split and in operand order from the caller (kept in step by the Adam kernel), the activations are split when they are
// made.  Layers 0 and 1 and g1 are computed transposed -- output columns on the accumulator's rows, batch rows on its
// columns -- so that a lane holds four consecutive columns of one batch row: it writes them as one 16-byte (bf16: 8-byte)
// piece, and they are the B operand of the head's product without a move.  dh1 is computed the other way round, where the
// accumulator is the B operand of dW0 = x^T g0.
//
// What bounds it: the chain of phases of one tile (a minibatch of 4096 gives every CU one tile of 32 rows), that is the
// latencies of the operand loads, of the loss (two exponentials and two logarithms in double precision) and of six
// barriers; matrix time is about a third.  More wavefronts per tile and 16-row tiles where they still fit the chip in
// one go make every phase shorter.  Per minibatch (all launches), against the form with 32-row tiles of two (H = 64) to
// eight wavefronts, fp32 matrix instructions and W1 staged through LDS: H = 64 28 -> 14 us (256 rows), 31.5 -> 20.6 us
// (4096 rows); H = 128 31.5 -> 17.6 us (256 rows); H = 256 56 -> 34 us (256 rows), 67.8 -> 50.4 us (4096 rows).
#include "mrl_host.hpp"
#include "mrl_device.hpp"
#include "mlp_tile.hpp"
#include "mlp_split.hpp"
#include "mlp3.hpp"
#include "mlp_rows16.hpp"
#include "ppo_grads.hpp"

namespace mrl {

struct DwFrag {
    int n;        // nets
    const unsigned short *x[2], *g[2];
    int off[2];   // of the net's W1 gradient in a split's partial vector
    const int32_t *skip;   // as FwdLoss::skip, never null
};

template <int H, int ACT, int RT>
__global__ __launch_bounds__(fb_threads(H)) void mlp3_fb_kernel(int B, int IN, Mlp3Nets nets, FwdLoss fl) {
    constexpr int T = fb_threads(H), NW = T / 64, NT = H / 16 / NW, R = 16 * RT, KS = H / 32;
    // (row pitches that spread a wavefront's 4-, 8- and 16-byte accesses over the LDS banks)
    constexpr int XLD = PIN_MAX + 1, PLD = H + 8, FLD = H + 20, GLD = 2 * PA_MAX + 1;
    constexpr int K0 = PIN_MAX / 4;
    constexpr int PF = KS < 3 ? KS : 3;          // k-steps of hidden-layer weights requested ahead
    constexpr bool DW_IN_TILE = H <= 128;        // (when the caller asks for it)
    constexpr bool BATCH_OPERANDS = H > 64 && NT % (2 / RT) == 0;   // (where the caller may ask for the weight-gradient launch)
    static_assert(R * 8 <= T && (H == 64 || R * 8 < T), "eight loss lanes per row; wavefronts left to store h1 where it is stored");
    __shared__ __align__(16) float xs[R * XLD];
    __shared__ __align__(16) __bf16 pieces[SPLIT][R * PLD];   // h1 going forward, g1 going back
    __shared__ __align__(16) float h1f[R * FLD];
    __shared__ __align__(16) float h2f[R * FLD];
    // (g1 lies over h2: a wavefront writes only columns whose h2 it alone reads, after it has read them)
    float *g1f = h2f;
    __shared__ __align__(16) float w2s[HEAD_LDS(H)];
    __shared__ float red[NW * R * (PA_MAX + 1)];
    __shared__ float g2s[R * GLD];
    const Mlp3Net nn = nets.n[blockIdx.y];
    const float *__restrict__ params = nn.params;
    const int A = nn.A;
    const bool GAUSS = nn.gauss != 0;
    const int ld = GAUSS ? 2 * A : A;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, g = lane >> 4, n = lane & 15;
    const long row0 = (long)blockIdx.x * R;
    const int nrow = (int)min((long)R, B - row0);
    float *__restrict__ db_part = nn.db_part + (size_t)blockIdx.x * (2 * H + PA_MAX);
    float *__restrict__ thin_part = nn.thin_part + (size_t)blockIdx.x * (size_t)nn.thin_stride;
    const bool actor = blockIdx.y == 0;

    // ---- Everything that does not depend on an earlier phase is requested first, the rows' indices (sixteen lanes a row;
    // the loss: eight) ahead of everything.  A lane past the last row, input or output asks for the last one's
    // value and drops it when it is used: behind a branch of its own every request would be waited for.
    const int skip = *fl.skip;   // (tested once these requests are out)
    constexpr int XQ = (R * 16 + T - 1) / T;
    const int32_t *__restrict__ idx = fl.idx + row0;
    int xsrc[XQ];
#pragma unroll
    for (int q = 0; q < XQ; ++q) xsrc[q] = idx[min((t + q * T) >> 4, nrow - 1)];
    const int lr = t >> 3, lj = t & 7;           // loss lanes: eight per row
    const bool loss_row = lr < nrow && t < 8 * R;
    const int lsrc = idx[min(lr, nrow - 1)];
    const float *lp_a = actor ? fl.r_adv : fl.r_ret, *lp_b = actor ? fl.r_logp : fl.r_val;
    const float *stats = fl.adv_stats != nullptr ? fl.adv_stats : fl.r_adv;    // (of the advantages; or any place with a value)
    const int act_w = fl.continuous ? fl.A : 1;
    float w0[NT][K0];
    f32x4 bias0[NT], bias1[NT];
    {
        const float *W0 = params, *b0 = params + IN * H, *b1 = b0 + H + H * H;
#pragma unroll
        for (int q = 0; q < NT; ++q) {
            const int c = 16 * (NT * w + q);
#pragma unroll
            for (int s = 0; s < K0; ++s)
                if (s == 0 || 4 * s < IN) w0[q][s] = W0[min(4 * s + g, IN - 1) * H + c + n];
            bias0[q] = *reinterpret_cast<const f32x4 *>(b0 + c + 4 * g);
            bias1[q] = *reinterpret_cast<const f32x4 *>(b1 + c + 4 * g);
        }
    }
    HeadLoads<H, T> head;
    const float *W2 = params + IN * H + H + H * H + H;
    head.load(W2, A, GAUSS, t);
    const float l_mean = stats[0], l_std = stats[fl.adv_stats != nullptr ? 1 : 0];
    float ls = W2[(H + (GAUSS ? 1 : 0)) * A + min(lj, A - 1)];    // log_std (no Gaussian head: a bias, not used)
    __builtin_amdgcn_sched_barrier(0);
    float xa[XQ], xb[XQ];
#pragma unroll
    for (int q = 0; q < XQ; ++q) {
        const float *x = fl.r_obs + (size_t)xsrc[q] * IN;
        const int j = t & 15;
        xa[q] = x[min(j, IN - 1)];
        xb[q] = x[min(j + 16, IN - 1)];
    }
    // critic: return, old value; actor: advantage, log-prob, action (component)
    const float l_a = lp_a[lsrc], l_b = lp_b[lsrc], l_act = fl.r_act[(size_t)lsrc * act_w + min(lj, act_w - 1)];
    if (skip != 0) return;
    __builtin_amdgcn_sched_barrier(0);
    bf16x8 wq[PF][NT][SPLIT];
    auto fetch = [&](const unsigned short *__restrict__ src, int ks, bf16x8 (&dst)[NT][SPLIT]) {
#pragma unroll
        for (int q = 0; q < NT; ++q)
#pragma unroll
            for (int p = 0; p < SPLIT; ++p)
                dst[q][p] = *reinterpret_cast<const bf16x8 *>(src + split_frag<H>(ks, NT * w + q, p, lane));
    };
    // under the wait for the rows: the head into LDS, and what of the loss needs no output
    if (blockIdx.x == 0 && actor)
        for (int i = t; i < fl.n_posts; i += T) fl.posts[i] = 0;
    for (int i = t; i < R * GLD; i += T) g2s[i] = 0.0f;
    head.store(w2s, A, GAUSS, t);
    const float std = actor && fl.continuous && t < 8 * R ? gaussian_std(ls, lj < A) : 1.0f;
#pragma unroll
    for (int q = 0; q < XQ; ++q) {
        const int r = (t + q * T) >> 4, j = t & 15;
        if (r < R) {
            if (j < IN) xs[r * XLD + j] = r < nrow ? xa[q] : 0.0f;
            if (j + 16 < IN) xs[r * XLD + j + 16] = r < nrow ? xb[q] : 0.0f;
            if (j == 0) xs[r * XLD + IN] = 1.0f;     // the bias gradient of layer 0 as row IN of x^T g0
        }
    }
    // (the weights last: another wavefront's rows would wait behind them)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < PF; ++i) fetch(nn.wf, i, wq[i]);
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();

    // ---- layer 0, transposed: D[column 4 g + v][batch row n]
    {
        float x[RT][K0];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int s = 0; s < K0; ++s)
                x[rt][s] = 4 * s + g < IN ? xs[(16 * rt + n) * XLD + 4 * s + g] : 0.0f;
        f32x4 d[NT][RT];
#pragma unroll
        for (int q = 0; q < NT; ++q)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) d[q][rt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < K0; ++s) {
            if (4 * s < IN) {
#pragma unroll
                for (int q = 0; q < NT; ++q)
#pragma unroll
                    for (int rt = 0; rt < RT; ++rt)
                        d[q][rt] = __builtin_amdgcn_mfma_f32_16x16x4f32(4 * s + g < IN ? w0[q][s] : 0.0f, x[rt][s], d[q][rt], 0, 0, 0);
            }
        }
#pragma unroll
        for (int q = 0; q < NT; ++q) {
            const int c = 16 * (NT * w + q) + 4 * g;
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const int r = 16 * rt + n;
                f32x4 y;
#pragma unroll
                for (int v = 0; v < 4; ++v) y[v] = activate<ACT>(d[q][rt][v] + bias0[q][v]);
                *reinterpret_cast<f32x4 *>(h1f + r * FLD + c) = y;
                bf16x4 p[SPLIT];
                split4(y, p);
#pragma unroll
                for (int i = 0; i < SPLIT; ++i) *reinterpret_cast<bf16x4 *>(&pieces[i][r * PLD + c]) = p[i];
            }
        }
    }
    __syncthreads();

    // ---- layer 1, transposed
    f32x4 h2v[RT][NT];
    {
        f32x4 hi[RT][NT], lo[RT][NT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int q = 0; q < NT; ++q) hi[rt][q] = lo[rt][q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            bf16x8 act[RT][SPLIT];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int p = 0; p < SPLIT; ++p)
                    act[rt][p] = *reinterpret_cast<const bf16x8 *>(&pieces[p][(16 * rt + n) * PLD + 32 * ks + 8 * g]);
#pragma unroll
            for (int q = 0; q < NT; ++q)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) mfma_split(wq[ks % PF][q], act[rt], hi[rt][q], lo[rt][q]);
            if (ks + PF < KS) fetch(nn.wf, ks + PF, wq[ks % PF]);
            __builtin_amdgcn_sched_barrier(0);   // (the next weights stay ahead of the products that hide them)
        }
        // the way back's first weights, requested here so that the loss hides them
#pragma unroll
        for (int i = 0; i < PF; ++i) fetch(nn.wb, i, wq[i]);
#pragma unroll
        for (int q = 0; q < NT; ++q) {
            const int c = 16 * (NT * w + q) + 4 * g;
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
                for (int v = 0; v < 4; ++v) h2v[rt][q][v] = activate<ACT>(split_sum(hi[rt][q][v], lo[rt][q][v]) + bias1[q][v]);
                *reinterpret_cast<f32x4 *>(h2f + (16 * rt + n) * FLD + c) = h2v[rt][q];
            }
        }
        // head: this wavefront's columns' share of out^T[a][row]; k-slot g of step v is column 4 g + v
        float a[NT][4];
#pragma unroll
        for (int q = 0; q < NT; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                a[q][v] = n < PA_MAX ? w2s[(16 * (NT * w + q) + 4 * g + v) * PA_MAX + n] : 0.0f;
        f32x4 d[RT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) d[rt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int q = 0; q < NT; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt)
                    d[rt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[q][v], h2v[rt][q][v], d[rt], 0, 0, 0);
        if (g < PA_MAX / 4) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int v = 0; v < 4; ++v) red[(w * R + 16 * rt + n) * (PA_MAX + 1) + 4 * g + v] = d[rt][v];
        }
    }
    __syncthreads();

    // ---- loss gradients, eight lanes per row: lane lj on output lj
    if (t < 8 * R) {
        float mine = 0.0f;
#pragma unroll
        for (int k = 0; k < NW; ++k) mine += red[(k * R + lr) * (PA_MAX + 1) + lj];
        mine += w2s[HEAD_B2(H) + lj];
        const long b = row0 + lr;
        float *g2row = g2s + lr * GLD;
        if (loss_row && lj < A) nn.out[b * ld + lj] = mine;
        if (!actor) {
            if (loss_row && lj == 0) {
                const float gv = critic_grad_value(mine, l_b, l_a, fl.mb, fl.continuous, fl.clip_value, fl.value_coef,
                                                   fl.clip_eps);
                g2row[0] = gv;
                fl.g_values[b] = gv;
            }
        } else {
            // (rows past nrow are worked on like the others -- their lanes take part in the exchanges -- and not stored)
            float adv = l_a, kl;
            if (fl.adv_stats != nullptr) adv = (adv - l_mean) / (l_std + 1e-8f);
            if (fl.continuous) {
                if (loss_row && lj < A)   // state-independent log_std, clamped (stochastic_actor.mojo:260-275)
                    nn.out[b * ld + A + lj] = ls < -5.0f ? -5.0f : (ls > 2.0f ? 2.0f : ls);
                float gm, gs;
                kl = actor_grad_gaussian_lanes(mine, ls, std, l_act, lj, lane & ~7, adv, l_b, fl.mb, A, fl.clip_eps,
                                               fl.ent_coef, gm, gs);
                if (loss_row && lj < A) {
                    g2row[lj] = gm;
                    g2row[A + lj] = gs;
                    fl.g_actor_out[b * ld + lj] = gm;
                    fl.g_actor_out[b * ld + A + lj] = gs;
                }
            } else {
                float gl;
                kl = actor_grad_discrete_lanes(mine, lj, lane & ~7, (int)l_act, adv, l_b, fl.mb, A, fl.clip_eps, fl.ent_coef,
                                               gl);
                if (loss_row && lj < A) {
                    g2row[lj] = gl;
                    fl.g_actor_out[b * ld + lj] = gl;
                }
            }
            if (loss_row && lj == 0) {
                fl.kl[b] = kl;
                g2row[2 * PA_MAX] = kl;   // (the spare float of the row, for the tile's sum below)
            }
        }
    } else if (BATCH_OPERANDS && !fl.dw_in_tiles) {
        // the wavefronts without loss rows: h1 out to the weight-gradient launch
        for (int ct = (w - R / 8) * (2 / RT); ct < H / 16; ct += (NW - R / 8) * (2 / RT)) batch_operand<H, RT, FLD>(h1f, nn.h1q, ct, lane);
    }
    __syncthreads();

    // ---- back through the head and layer 1's activation: g1^T, on the lanes that hold h2
    {
        float w2[NT][PA_MAX / 4], gb[RT][PA_MAX / 4], gr[4 * RT];
#pragma unroll
        for (int s = 0; s < PA_MAX / 4; ++s) {
#pragma unroll
            for (int q = 0; q < NT; ++q) w2[q][s] = w2s[(16 * (NT * w + q) + n) * PA_MAX + 4 * s + g];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) gb[rt][s] = g2s[(16 * rt + n) * GLD + 4 * s + g];
        }
#pragma unroll
        for (int s = 0; s < 4 * RT; ++s) gr[s] = g2s[(4 * s + g) * GLD + n];
        f32x4 d[NT][RT], d2[NT];
#pragma unroll
        for (int q = 0; q < NT; ++q) {
            d2[q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) d[q][rt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
#pragma unroll
        for (int s = 0; s < PA_MAX / 4; ++s)   // (W2's rows are zero beyond A)
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
#pragma unroll
        for (int q = 0; q < NT; ++q) {
            const int c = 16 * (NT * w + q) + 4 * g;
            f32x4 cs = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const int r = 16 * rt + n;
                f32x4 y;
#pragma unroll
                for (int v = 0; v < 4; ++v) y[v] = d[q][rt][v] * act_deriv_out<ACT>(h2v[rt][q][v]);
                cs = cs + y;
                bf16x4 p[SPLIT];
                split4(y, p);
#pragma unroll
                for (int i = 0; i < SPLIT; ++i) *reinterpret_cast<bf16x4 *>(&pieces[i][r * PLD + c]) = p[i];
                *reinterpret_cast<f32x4 *>(g1f + r * FLD + c) = y;
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
        if (BATCH_OPERANDS && !fl.dw_in_tiles) {
            // g1 out to the weight-gradient launch (its columns were written by this wavefront)
            asm volatile("" : : : "memory");
#pragma unroll
            for (int q = 0; q < NT; q += 2 / RT) batch_operand<H, RT, FLD>(g1f, nn.g1q, NT * w + q, lane);
        }
    }
    if (w == NW - 1 && lane < ld) {   // column sums of the tile: bias gradient of the head, log_std gradient
        float s = 0.0f;
#pragma unroll
        for (int r = 0; r < R; ++r) s += g2s[r * GLD + lane];
        if (lane < A) db_part[2 * H + lane] = s;
        else nn.ls_part[(long)blockIdx.x * A + (lane - A)] = s;
    }
    if (w == NW - 2 && actor && fl.kl_flag != nullptr) {
        // KL test: every actor tile leaves the sum of its rows' estimates; the kernel that applies the update adds the
        // tiles up and compares the mean with target_kl, so that nothing here waits for other workgroups
        float kl = lane < nrow ? g2s[(lane < R ? lane : 0) * GLD + 2 * PA_MAX] : 0.0f;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) kl += __shfl_xor(kl, off, 64);
        if (lane == 0) fl.kl_part[blockIdx.x] = kl;
    }
    __syncthreads();

    // ---- dh1 = g1 W1^T: D[batch row 4 g + v][column n]
    {
        f32x4 hi[RT][NT], lo[RT][NT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int q = 0; q < NT; ++q) hi[rt][q] = lo[rt][q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            bf16x8 a[RT][SPLIT];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int p = 0; p < SPLIT; ++p)
                    a[rt][p] = *reinterpret_cast<const bf16x8 *>(&pieces[p][(16 * rt + n) * PLD + 32 * ks + 8 * g]);
#pragma unroll
            for (int q = 0; q < NT; ++q)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) mfma_split(a[rt], wq[ks % PF][q], hi[rt][q], lo[rt][q]);
            if (ks + PF < KS) fetch(nn.wb, ks + PF, wq[ks % PF]);
            __builtin_amdgcn_sched_barrier(0);
        }
        float g0[NT][RT][4];
#pragma unroll
        for (int q = 0; q < NT; ++q)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    g0[q][rt][v] = split_sum(hi[rt][q][v], lo[rt][q][v]) *
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
    }
    if constexpr (DW_IN_TILE) {
        // The hidden layer's weight gradient of the tile, dW1[k][c] = sum over rows of h1[row][k] g1[row][c], as one more
        // per-tile piece for the sum kernel, instead of in a launch of its own that reads h1 and g1 back from global
        // memory, where the launch is the larger part (dw_in_tiles_pays).
        if (fl.dw_in_tiles) {
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
}

// dW = h1^T g1 of the hidden layer of one or two nets over a split of the batch: partial[split][Ptot].  Operands as the row
// tiles left them (split, in operand order), straight from global memory into registers: no LDS, no barrier.  A
// workgroup makes one 64 x 128 output tile (four wavefronts, 32 x 64 each) twice over, two groups of wavefronts taking
// alternate k-steps of 32 batch rows and adding up at the end.
// What bounds it: fetching the operands (25 MB at a minibatch of 4096, written by the launch before), then the matrix
// cores (48 instructions of 16 cycles per wavefront and k-step; a k-step's operands are in flight while the one before
// is multiplied).  256 rows per split give every CU one workgroup at a minibatch of 4096 and
// H = 256; more splits would be more partial sums to write and read back.  H = 256, 4096 rows, both nets: 12.6 us, against
// 16.1 us with fp32 matrix instructions and 16.3 us when every workgroup splits its fp32 rows itself.
// Workgroups go to the chip's eight XCDs in turn, and each XCD has an L2 of its own: the tiles of one (net, split) read
// the same rows, so the flat list of workgroups gives them to ONE XCD.
template <int H>
__global__ __launch_bounds__(512) void dw_frag_kernel(DwFrag d, int steps, int steps_per, int splits, int Ptot,
                                                      float *__restrict__ partial) {
    const int skip = *d.skip;
    __builtin_amdgcn_sched_barrier(0);
    constexpr int XCDS = 8, TN = 128, tiles_n = H / TN, tiles = tiles_n * (H / 64), NB = 4, RLD = TN + 4;
    static_assert(H % TN == 0, "whole tiles");
    __shared__ float sum[64 * RLD];
    const int groups = d.n * splits;
    // workgroup n = (round r, XCD x): the r-th workgroup that XCD x receives.  An XCD walks its groups x, x + 8, ... one
    // after the other, `tiles` workgroups each; the workgroups of a short last round keep the plain order.
    int grp, tile;
    {
        const int nwg = blockIdx.x, full = (groups / XCDS) * XCDS * tiles;
        const int x = nwg % XCDS, q = nwg / XCDS, m = nwg - full;
        tile = nwg < full ? q % tiles : m % tiles;
        grp = nwg < full ? (q / tiles) * XCDS + x : (groups / XCDS) * XCDS + m / tiles;
    }
    const int net = grp / splits, z = grp % splits;
    const int t = threadIdx.x, lane = t & 63, half = t >> 8, wr = (t >> 7) & 1, wc = (t >> 6) & 1, g = lane >> 4, n = lane & 15;
    const int ct_a = (tile / tiles_n) * 4 + 2 * wr, ct_b = (tile % tiles_n) * (TN / 16) + NB * wc;
    const int k0 = z * steps_per + half, k1 = min(z * steps_per + steps_per, steps);
    const unsigned short *__restrict__ X = d.x[net], *__restrict__ G = d.g[net];
    f32x4 hi[2][NB], lo[2][NB];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b) hi[a][b] = lo[a][b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    bf16x8 fa[2][2][SPLIT], fb[2][NB][SPLIT];   // [buffer]
    auto fetch = [&](int ks, int u) {
#pragma unroll
        for (int q = 0; q < SPLIT; ++q) {
#pragma unroll
            for (int a = 0; a < 2; ++a) fa[u][a][q] = *reinterpret_cast<const bf16x8 *>(X + split_frag<H>(ks, ct_a + a, q, lane));
#pragma unroll
            for (int b = 0; b < NB; ++b) fb[u][b][q] = *reinterpret_cast<const bf16x8 *>(G + split_frag<H>(ks, ct_b + b, q, lane));
        }
    };
    auto multiply = [&](int u) {
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int a = 0; a < 2; ++a) mfma_split(fa[u][a], fb[u][b], hi[a][b], lo[a][b]);
    };
    if (k0 < k1) fetch(k0, 0);
    if (skip != 0) return;
    for (int k = k0; k < k1; k += 4) {   // two k-steps per round, so that the buffers keep their names
        if (k + 2 < k1) fetch(k + 2, 1);
        __builtin_amdgcn_sched_barrier(0);
        multiply(0);
        if (k + 2 < k1) {
            if (k + 4 < k1) fetch(k + 4, 0);
            __builtin_amdgcn_sched_barrier(0);
            multiply(1);
        }
    }
    if (half == 1) {
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    sum[(32 * wr + 16 * a + 4 * g + v) * RLD + 64 * wc + 16 * b + n] = split_sum(hi[a][b][v], lo[a][b][v]);
    }
    __syncthreads();
    if (half == 1) return;
    float *out = partial + (size_t)z * Ptot + d.off[net] + (size_t)(tile / tiles_n) * 64 * H + (tile % tiles_n) * TN;
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int r = 32 * wr + 16 * a + 4 * g + v, c = 64 * wc + 16 * b + n;
                out[(size_t)r * H + c] = sum[r * RLD + c] + split_sum(hi[a][b][v], lo[a][b][v]);
            }
}

// P0: parameters of the first net, w1_off: offset of W1 in a net's parameters
int launch_dw_frag(mrl_ctx *ctx, int H, int n_nets, int batch, const UpdateWs &ws, int P0, int Ptot, int w1_off,
                   const int32_t *skip) {
    DwFrag d{};
    d.n = n_nets;
    d.skip = skip;
    for (int i = 0; i < n_nets; ++i) {
        d.x[i] = ws.net[i].h1q;
        d.g[i] = ws.net[i].g1q;
        d.off[i] = (i ? P0 : 0) + w1_off;
    }
    const int steps = (batch + 31) / 32;
    const dim3 grid(n_nets * ws.splits * (H / 64) * (H / 128)), block(512);
    if (H == 256) hipLaunchKernelGGL(dw_frag_kernel<256>, grid, block, 0, ctx->stream, d, steps, ws.steps_per, ws.splits, Ptot, ws.partial);
    else if (H == 128) hipLaunchKernelGGL(dw_frag_kernel<128>, grid, block, 0, ctx->stream, d, steps, ws.steps_per, ws.splits, Ptot, ws.partial);
    else return MRL_E_UNSUPPORTED;
    MRL_CHECK_LAUNCH();
    return MRL_OK;
}

// Split operand copies of the hidden layer's weights of one or two nets, both orientations; grid = (H * H / 8 / 256
// (at least one), orientations, nets)
template <int H>
__global__ __launch_bounds__(256) void split_weights_kernel(SplitNets s) {
    const int e = blockIdx.x * 256 + threadIdx.x, net = blockIdx.z;
    if (e >= H * H / 8) return;
    const float *__restrict__ W = s.w1[net];
    f32x8 x;
    int k8, other;    // eight consecutive values of the contracted index, the other index
    if (blockIdx.y == 0) {
        k8 = e / H; other = e % H;
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = W[(size_t)(8 * k8 + j) * H + other];
    } else {
        other = e / (H / 8); k8 = e % (H / 8);
        const f32x4 a = *reinterpret_cast<const f32x4 *>(W + (size_t)other * H + 8 * k8);
        const f32x4 b = *reinterpret_cast<const f32x4 *>(W + (size_t)other * H + 8 * k8 + 4);
#pragma unroll
        for (int j = 0; j < 4; ++j) { x[j] = a[j]; x[4 + j] = b[j]; }
    }
    bf16x8 p[SPLIT];
    split8(x, p);
    unsigned short *dst = blockIdx.y == 0 ? s.wf[net] : s.wb[net];
#pragma unroll
    for (int i = 0; i < SPLIT; ++i)
        *reinterpret_cast<bf16x8 *>(dst + split_frag<H>(k8 >> 2, other >> 4, i, (k8 & 3) * 16 + (other & 15))) = p[i];
}

template <int H>
static void launch_split(hipStream_t st, const SplitNets &s, int n_nets) {
    hipLaunchKernelGGL(split_weights_kernel<H>, dim3((H * H / 8 + 255) / 256, 2, n_nets), dim3(256), 0, st, s);
}
int launch_split_weights(mrl_ctx *ctx, int H, const SplitNets &s, int n_nets) {
    if (H == 256) launch_split<256>(ctx->stream, s, n_nets);
    else if (H == 128) launch_split<128>(ctx->stream, s, n_nets);
    else launch_split<64>(ctx->stream, s, n_nets);
    MRL_CHECK_LAUNCH();
    return MRL_OK;
}

template <int H, int ACT>
static void launch_fb_t(mrl_ctx *ctx, int batch, int IN, int rows, const Mlp3Nets &nets, const FwdLoss &fl) {
    const dim3 grid((batch + rows - 1) / rows, 2), block(fb_threads(H));
    if (rows == 16) hipLaunchKernelGGL((mlp3_fb_kernel<H, ACT, 1>), grid, block, 0, ctx->stream, batch, IN, nets, fl);
    else hipLaunchKernelGGL((mlp3_fb_kernel<H, ACT, 2>), grid, block, 0, ctx->stream, batch, IN, nets, fl);
}
int launch_fb(mrl_ctx *ctx, int H, int act, int batch, int IN, int rows, const Mlp3Nets &nets, const FwdLoss &fl) {
    if (H == 256 && act == 1) launch_fb_t<256, 1>(ctx, batch, IN, rows, nets, fl);
    else if (H == 256) launch_fb_t<256, 2>(ctx, batch, IN, rows, nets, fl);
    else if (H == 128 && act == 1) launch_fb_t<128, 1>(ctx, batch, IN, rows, nets, fl);
    else if (H == 128) launch_fb_t<128, 2>(ctx, batch, IN, rows, nets, fl);
    else if (act == 1) launch_fb_t<64, 1>(ctx, batch, IN, rows, nets, fl);
    else launch_fb_t<64, 2>(ctx, batch, IN, rows, nets, fl);
    MRL_CHECK_LAUNCH();
    return MRL_OK;
}

}  // namespace mrl
