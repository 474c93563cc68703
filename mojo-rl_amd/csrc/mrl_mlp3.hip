// The fused passes over three-layer nets  IN -> H -> H -> out  (H in {64, 128, 256}, IN <= 32, out <= 8 or a
// StochasticActor head of <= 8 actions): the shapes of every actor and critic the PPO agents build
// (deep_agents/ppo/ppo.mojo:779-817, ppo_continuous.mojo:171-194).
//
//   mlp3_fwd_kernel     the whole forward of a 32-row tile in one launch (hidden activations
//                       stay in LDS), writing the reference's per-layer cache on the way, for batches
//                       beyond those that the 16-row tiles of mrl_rows.hip take;
//   sum3_kernel         sum of the batch splits and of the row tiles' pieces straight into the flat gradient vector;
// and the host side of these, of the backward (mrl_rows.hip) and of the minibatch update (mrl_fb.hip).  The per-layer
// kernels (mrl_mlp.hip) remain the path for any other shape.
#include "mrl_host.hpp"
#include "mrl_device.hpp"
#include "mlp_tile.hpp"
#include "mlp_split.hpp"
#include "mlp3.hpp"
#include "tile_sums.hpp"

namespace mrl {

// grid = row tiles
template <int H, int ACT>
__global__ __launch_bounds__(2 * H) void mlp3_fwd_kernel(int B, int IN, Mlp3Net nn) {
    constexpr int T = 2 * H;   // one 32-column accumulator tile per wavefront
    __shared__ float xs[PR * XS_LD];
    __shared__ float hT[H * HT_LD];
    __shared__ float h2[PR * (H + 1)];
    __shared__ float ys[PR * (PA_MAX + 1)];
    __shared__ __align__(16) float w2s[HEAD_LDS(H)];
    const float *__restrict__ x = nn.x;
    const float *__restrict__ params = nn.params;
    float *__restrict__ out = nn.out;
    float *__restrict__ cache = nn.cache;
    const int A = nn.A;
    const bool GAUSS = nn.gauss != 0;
    const int t = threadIdx.x;
    const long row0 = (long)blockIdx.x * PR;
    const int nrow = (int)min((long)PR, B - row0);
    TileCache tc{nullptr, nullptr, nullptr, row0, nrow};
    if (cache != nullptr) {
        tc.c0 = cache;
        tc.c1 = cache + (size_t)B * (IN + H);
        tc.c2 = tc.c1 + (size_t)B * 2 * H;
    }
    // every load that does not depend on an earlier phase goes out first
    HiddenOperands<H, 1, 32> ops;
    ops.load(params, IN);
    constexpr int NX = (PR * PIN_MAX + T - 1) / T;
    float xv[NX];
#pragma unroll
    for (int q = 0; q < NX; ++q) {
        const int i = t + q * T;
        xv[q] = 0.0f;
        if (i < PR * IN && i / IN < nrow) {
            xv[q] = x[row0 * IN + i];
        }
    }
    stage_head(params + IN * H + H + H * H + H, H, A, GAUSS, w2s, t, T);
#pragma unroll
    for (int q = 0; q < NX; ++q) {
        const int i = t + q * T;
        if (i < PR * IN) {
            const int r = i / IN, k = i - r * IN;
            xs[r * XS_LD + k] = xv[q];
            if (r < nrow && cache != nullptr) tc.c0[(row0 + r) * (IN + H) + k] = xv[q];
        }
    }
    __syncthreads();
    hidden_stack<H, ACT, 1>(params, IN, xs, hT, h2, tc, ops);
    head<H>(w2s, A, h2, ys, PA_MAX + 1, t, 2 * H);
    __syncthreads();
    const int ld = GAUSS ? 2 * A : A;
    for (int i = t; i < nrow * ld; i += T) {
        const int r = i / ld, a = i - r * ld;
        float v;
        if (a < A) {
            v = ys[r * (PA_MAX + 1) + a];
        } else {   // state-independent log_std, clamped (deep_rl/model/stochastic_actor.mojo:260-275)
            v = w2s[HEAD_LOG_STD(H) + (a - A)];
            if (v < -5.0f) v = -5.0f;
            else if (v > 2.0f) v = 2.0f;
        }
        out[(row0 + r) * ld + a] = v;
    }
}

template <bool TREE>
__global__ __launch_bounds__(256) void sum3_kernel(SumNets sn, float *__restrict__ sq_part) {
    const int skip = *sn.skip;
    __builtin_amdgcn_sched_barrier(0);
    __shared__ float red[2][4];
    const int gi = blockIdx.x * blockDim.x + threadIdx.x;
    const int P0 = sn.net[0].P, net = sn.n > 1 && gi >= P0 ? 1 : 0, i = gi - (net ? P0 : 0);
    float s = 0.0f;
    if (i < sn.net[net].P) {
        const int o1 = (sn.IN + 1) * sn.H, HH = sn.H * sn.H;
        const SumTerms inner = hidden_terms(sn.net[net], i - o1), outer = thin_terms(sn.net[net], sn.IN, sn.H, sn.tiles, i);
        const bool in = i >= o1 && i < o1 + HH;
        if (skip == 0) {
            s = sum_terms<TREE, float>({in ? inner.p : outer.p, in ? inner.stride : outer.stride, in ? inner.n : outer.n});
            sn.net[net].grads[i] = s;
        }
    }
    if (sq_part == nullptr) return;
    // per-block sums of squares, one per net (a block may straddle the two vectors): the partials
    // of the global-norm clip, sq_part[net * 1024 + block]
    float v0 = net == 0 ? s * s : 0.0f, v1 = net == 1 ? s * s : 0.0f;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        v0 += __shfl_xor(v0, off, 64);
        v1 += __shfl_xor(v1, off, 64);
    }
    if ((threadIdx.x & 63) == 0) { red[0][threadIdx.x >> 6] = v0; red[1][threadIdx.x >> 6] = v1; }
    __syncthreads();
    if (threadIdx.x < 2) {
        const float *r = red[threadIdx.x];
        sq_part[threadIdx.x * 1024 + blockIdx.x] = r[0] + r[1] + r[2] + r[3];
    }
}

// ---------------------------------------------------------------- host side

bool mlp3_fusable(const mrl_mlp_desc &d, int *H, int *act, bool *gauss) {
    if (d.n_layers != 3) return false;
    const int k0 = d.layers[0].kind;
    if ((k0 != MRL_LINEAR_RELU && k0 != MRL_LINEAR_TANH) || d.layers[1].kind != k0) return false;
    const int k2 = d.layers[2].kind;
    if (k2 != MRL_LINEAR && k2 != MRL_STOCHASTIC_ACTOR) return false;
    const int h = d.layers[0].out_dim;
    if ((h != 64 && h != 128 && h != 256) || d.layers[1].out_dim != h) return false;
    if (d.layers[0].in_dim > PIN_MAX || d.layers[2].out_dim > PA_MAX) return false;
    *H = h;
    *act = k0 == MRL_LINEAR_RELU ? 1 : 2;
    *gauss = k2 == MRL_STOCHASTIC_ACTOR;
    return true;
}

static int net_P(const mrl_mlp_desc &d) {
    const int IN = d.layers[0].in_dim, H = d.layers[0].out_dim, A = d.layers[2].out_dim;
    return (IN + 1) * H + (H + 1) * H + (H + 1) * A + (d.layers[2].kind == MRL_STOCHASTIC_ACTOR ? A : 0);
}

// Rows per tile of the fused update kernel: 16 while both nets' tiles fit the chip's CUs in one go, else 32 (a weight
// operand then serves two row tiles, and half as many per-tile pieces are added up).  us per minibatch of 256 / 1024 /
// 2048 / 4096 rows, 16 against 32: H = 64 14.0 / 15.5 / 17.8 / 23.3 : 18.1 / 17.7 / 18.0 / 20.6; H = 256 33.8 / 37.3 /
// 40.8 / 60.5 : 40.9 / 42.3 / 45.1 / 50.4; H = 128, whose pieces hold the H x H gradient as well, 17.6 / 21.9 / 26.5 /
// 33.3 : 22.9 / 23.1 / 25.8 / 29.9, hence half the bound there.
static int fb_tile_rows(int n_cus, int H, int n_nets, int batch) {
    return n_nets * ((batch + 15) / 16) <= (H == 128 ? n_cus / 2 : n_cus) ? 16 : 32;
}

// Whether the fused update kernel takes the hidden layer's weight gradient of its row tile itself
// (H^2 floats per tile and net, added up by the sum kernel) or leaves h1 and g1 to a launch of dw_frag_kernel.
static bool dw_in_tiles_pays(int H, int batch) { return H == 64 || (H == 128 && batch <= 8192); }

// true when the two nets can share launches: both fusable, same input width, width and activation
bool mlp3_pair_fusable(const mrl_mlp_desc &a, const mrl_mlp_desc &b) {
    int ha, hb, aa, ab;
    bool ga, gb;
    return mlp3_fusable(a, &ha, &aa, &ga) && mlp3_fusable(b, &hb, &ab, &gb) && ha == hb && aa == ab &&
           a.layers[0].in_dim == b.layers[0].in_dim;
}

// Whether the forward takes 16 rows per workgroup (mrl_rows.hip) or 32: 16 while a CU gets one workgroup at H = 256 (its
// eight wavefronts hold W1 in registers, a second one waits for them), two at H = 128, and as far as measured at H = 64.
// us, 16 against 32 rows, cache written, tanh, 24 inputs: H = 256 13.9 : 18.5 (33 rows), 17.7 : 20.9 (4096), 31.6 : 22.9
// (8191); H = 128 7.1 : 10.6 (33), 11.7 : 13.7 (8191), 18.5 : 18.3 (16384); H = 64 5.7 : 10.4 (33), 10.1 : 15.7 (16384).
static bool fwd_rows_16(int n_cus, int H, int batch) {
    return (batch + 15) / 16 <= (H == 256 ? 1 : H == 128 ? 2 : 16) * n_cus;
}

template <int H, int ACT>
static void launch_fwd_t(mrl_ctx *ctx, int batch, int IN, const Mlp3Net &nn) {
    hipLaunchKernelGGL((mlp3_fwd_kernel<H, ACT>), dim3((batch + PR - 1) / PR), dim3(2 * H), 0, ctx->stream, batch, IN, nn);
}
int mlp3_forward(mrl_ctx *ctx, const mrl_mlp_desc &d, int batch, const float *in, const float *params,
                 float *out, float *cache) {
    int H = 0, act = 0;
    bool gauss = false;
    if (!mlp3_fusable(d, &H, &act, &gauss)) return MRL_E_UNSUPPORTED;
    Mlp3Net nn{};
    nn.x = in; nn.params = params; nn.out = out; nn.cache = cache;
    nn.A = d.layers[2].out_dim;
    nn.gauss = gauss ? 1 : 0;
    const int IN = d.layers[0].in_dim;
    if (fwd_rows_16(ctx->n_cus, H, batch)) return launch_fwd16(ctx, H, act, batch, IN, nn);
    if (H == 256 && act == 1) launch_fwd_t<256, 1>(ctx, batch, IN, nn);
    else if (H == 256) launch_fwd_t<256, 2>(ctx, batch, IN, nn);
    else if (H == 128 && act == 1) launch_fwd_t<128, 1>(ctx, batch, IN, nn);
    else if (H == 128) launch_fwd_t<128, 2>(ctx, batch, IN, nn);
    else if (act == 1) launch_fwd_t<64, 1>(ctx, batch, IN, nn);
    else launch_fwd_t<64, 2>(ctx, batch, IN, nn);
    MRL_CHECK_LAUNCH();
    return MRL_OK;
}

// batch splits of the weight-gradient launch: slices of whole k-chunks
static void dw_splits(int n_nets, int batch, int *splits, int *rows_per) {
    int s = std::max(1, std::min(32, batch / (128 * n_nets)));
    *rows_per = ((batch + s - 1) / s + 31) / 32 * 32;
    *splits = (batch + *rows_per - 1) / *rows_per;
}

// where the pieces of a call's gradients lie
SumNets mlp3_sum_nets(const mrl_mlp_desc *const *descs, int n_nets, const UpdateWs &ws, float *const *grads, const int32_t *skip) {
    const int IN = descs[0]->layers[0].in_dim, H = descs[0]->layers[0].out_dim;
    SumNets sn{};
    sn.n = n_nets;
    sn.IN = IN;
    sn.skip = skip;
    sn.H = H;
    sn.tiles = ws.tiles;
    int Ptot = 0, at = 0;
    for (int i = 0; i < n_nets; ++i) Ptot += net_P(*descs[i]);
    for (int i = 0; i < n_nets; ++i) {
        const Mlp3Net &from = ws.net[i];
        SumNet &net = sn.net[i];
        net.grads = grads[i];
        net.ls = from.ls_part;
        net.db = from.db_part;
        net.thin = from.thin_part;
        net.thin_stride = from.thin_stride;
        net.P = net_P(*descs[i]);
        net.A = descs[i]->layers[2].out_dim;
        if (ws.dw_in_tiles) {   // behind dW0 and dW2 of every tile
            net.hidden = from.thin_part + (size_t)IN * H + (size_t)H * net.A;
            net.hidden_stride = from.thin_stride;
            net.hidden_n = ws.tiles;
        } else {                // the nets' vectors lie back to back in a split's
            net.hidden = ws.partial + at + (IN + 1) * H;
            net.hidden_stride = Ptot;
            net.hidden_n = ws.splits;
        }
        at += net.P;
    }
    return sn;
}

// The sums over row tiles and batch splits into the flat gradients.
int mlp3_sum_tiles(mrl_ctx *ctx, const SumNets &sn, int tile_rows, float *sq_part, int *sq_blocks) {
    const int sum_blocks = grid_for(sn.net[0].P + (sn.n > 1 ? sn.net[1].P : 0), 256);
    if (sum_blocks > 1024) sq_part = nullptr;   // more partials than the caller's buffer holds
    if (sq_blocks) *sq_blocks = sq_part ? sum_blocks : 0;
    if (tile_rows == 16) hipLaunchKernelGGL(sum3_kernel<true>, dim3(sum_blocks), dim3(256), 0, ctx->stream, sn, sq_part);
    else hipLaunchKernelGGL(sum3_kernel<false>, dim3(sum_blocks), dim3(256), 0, ctx->stream, sn, sq_part);
    MRL_CHECK_LAUNCH();
    return MRL_OK;
}

// carves (and if need be grows) the context's workspace for the fused update of two nets, or the backward of one (params
// null: no copies of the weights)
int mlp3_update_ws(mrl_ctx *ctx, const mrl_mlp_desc *const *descs, int n_nets, int batch, const float *const *params, UpdateWs *out) {
    const int H = descs[0]->layers[0].out_dim, IN = descs[0]->layers[0].in_dim;
    UpdateWs &u = *out;
    u = UpdateWs{};
    u.rows = fb_tile_rows(ctx->n_cus, H, n_nets, batch);
    u.tiles = (batch + u.rows - 1) / u.rows;
    u.dw_in_tiles = dw_in_tiles_pays(H, batch);
    int rows_per;
    dw_splits(n_nets, batch, &u.splits, &rows_per);
    u.steps_per = rows_per / 32;
    size_t need = 0, P = 0;
    float *base = nullptr;
    for (int pass = 0; pass < 2; ++pass) {   // sizes, then pointers (every piece a multiple of four floats)
        size_t at = 0;
        auto take = [&](size_t floats) {
            float *p = pass ? base + at : nullptr;
            at += (floats + 3) / 4 * 4;
            return p;
        };
        P = 0;
        for (int i = 0; i < n_nets; ++i) {
            const int A = descs[i]->layers[2].out_dim;
            if (params != nullptr) {
                u.split.w1[i] = params[i] + IN * H + H;
                u.split.wf[i] = reinterpret_cast<unsigned short *>(take(split_elems(H) / 2));
                u.split.wb[i] = reinterpret_cast<unsigned short *>(take(split_elems(H) / 2));
            }
            if (!u.dw_in_tiles) {
                const size_t elems = (size_t)SPLIT * ((batch + 31) / 32) * 32 * H;
                u.net[i].h1q = reinterpret_cast<unsigned short *>(take(elems / 2));
                u.net[i].g1q = reinterpret_cast<unsigned short *>(take(elems / 2));
            }
            u.net[i].ls_part = take((size_t)u.tiles * PA_MAX);
            u.net[i].db_part = take((size_t)u.tiles * (2 * H + PA_MAX));
            u.net[i].thin_stride = IN * H + H * A + (u.dw_in_tiles ? H * H : 0);
            u.net[i].thin_part = take((size_t)u.tiles * (size_t)u.net[i].thin_stride);
            P += net_P(*descs[i]);
        }
        u.partial = take(u.dw_in_tiles ? 4 : (size_t)u.splits * P);
        need = at;
        if (pass == 0) {
            int rc = mlp_ensure_ws(ctx, need, &base);
            if (rc) return rc;
        }
    }
    return MRL_OK;
}

int mlp3_update_n(mrl_ctx *ctx, const mrl_mlp_desc *const *descs, int batch, Mlp3Nets io, const UpdateWs &ws, const FwdLoss &loss) {
    int H = 0, act = 0;
    bool gauss = false;
    for (int i = 0; i < 2; ++i) {
        if (!mlp3_fusable(*descs[i], &H, &act, &gauss)) return MRL_E_UNSUPPORTED;
        Mlp3Net &nn = io.n[i];
        const Mlp3Net &from = ws.net[i];
        nn.A = descs[i]->layers[2].out_dim;
        nn.gauss = gauss ? 1 : 0;
        nn.g1q = from.g1q; nn.h1q = from.h1q; nn.ls_part = from.ls_part; nn.db_part = from.db_part;
        nn.thin_part = from.thin_part; nn.thin_stride = from.thin_stride;
        nn.wf = ws.split.wf[i]; nn.wb = ws.split.wb[i];
    }
    FwdLoss fl = loss;
    fl.dw_in_tiles = ws.dw_in_tiles ? 1 : 0;
    int rc = launch_fb(ctx, H, act, batch, descs[0]->layers[0].in_dim, ws.rows, io, fl);
    if (rc) return rc;
    if (!ws.dw_in_tiles) {
        const int P0 = net_P(*descs[0]);
        rc = launch_dw_frag(ctx, H, 2, batch, ws, P0, P0 + net_P(*descs[1]), (descs[0]->layers[0].in_dim + 1) * H, fl.skip);
        if (rc) return rc;
    }
    return MRL_OK;
}

// true when [a, a + na) and [b, b + nb) (floats) share memory
static bool overlap(const float *a, size_t na, const float *b, size_t nb) {
    const uintptr_t pa = reinterpret_cast<uintptr_t>(a), pb = reinterpret_cast<uintptr_t>(b);
    return pa < pb + 4 * nb && pb < pa + 4 * na;
}

// Backward of one net; MRL_E_UNSUPPORTED where the row tiles cannot take it: other shapes, parameters that 16-byte loads
// do not reach, and an input gradient that lies over something that other tiles still read.
int mlp3_backward(mrl_ctx *ctx, const mrl_mlp_desc &d, int batch, const float *grad_out, const float *params,
                  const float *cache, float *grads, float *grad_in) {
    int H = 0, act = 0;
    bool gauss = false;
    if (!mlp3_fusable(d, &H, &act, &gauss) || reinterpret_cast<uintptr_t>(params) % 16 != 0) return MRL_E_UNSUPPORTED;
    const int IN = d.layers[0].in_dim, A = d.layers[2].out_dim, P = net_P(d);
    const size_t n_in = (size_t)batch * IN;
    if (grad_in != nullptr &&
        (overlap(grad_in, n_in, grad_out, (size_t)batch * (gauss ? 2 * A : A)) || overlap(grad_in, n_in, params, P) ||
         overlap(grad_in, n_in, grads, P) || overlap(grad_in, n_in, cache, (size_t)batch * (IN + 4 * H))))
        return MRL_E_UNSUPPORTED;
    const mrl_mlp_desc *ds[1] = {&d};
    float *gs[1] = {grads};
    UpdateWs ws;
    int rc = mlp3_update_ws(ctx, ds, 1, batch, nullptr, &ws);
    if (rc) return rc;
    Mlp3Nets io{};
    Mlp3Net &nn = io.n[0];
    nn = ws.net[0];
    nn.A = A;
    nn.gauss = gauss ? 1 : 0;
    nn.grad_out = grad_out; nn.params = params; nn.cache = const_cast<float *>(cache); nn.grad_in = grad_in;
    rc = launch_bwd(ctx, H, act, batch, IN, ws.rows, nn, ws.dw_in_tiles);
    if (rc) return rc;
    if (!ws.dw_in_tiles) {
        rc = launch_dw_frag(ctx, H, 1, batch, ws, P, P, (IN + 1) * H, never_skip(ctx));
        if (rc) return rc;
    }
    return mlp3_sum_tiles(ctx, mlp3_sum_nets(ds, 1, ws, gs, never_skip(ctx)), ws.rows, nullptr, nullptr);
}

}  // namespace mrl
