// One PPO minibatch update -- the body of the minibatch loop of train_gpu
// (deep_agents/ppo/ppo.mojo:2438-2727, deep_agents/ppo/ppo_continuous.mojo:3000-3260) -- as one
// call that only enqueues: gather, per-minibatch advantage normalisation, actor and critic
// forward, loss gradients, KL test, backward, global-norm clip, Adam (and the log_std clamp).
// The actor and the critic do not depend on each other inside a minibatch, so when both have one
// of the fused shapes they run side by side in every launch, and a row tile never leaves its
// workgroup between the forward pass and the way back (mrl_fb.hip): 2 or 3 launches per minibatch (forward + loss
// gradients + KL test + backward; dW of the hidden layer, where the tiles do not leave it; sum + clip + Adam) instead
// of about 40.  The minibatch is not gathered: the forward reads its rows from the rollout through the indices and the loss
// normalises the advantage with statistics computed ahead (once per epoch for all minibatches).
// Other net shapes go layer by layer: gather + normalise, forward, loss gradients + KL test,
// backward, clip + Adam.
//
// KL early stop: the reference copies the per-sample KL to the host after the actor's loss
// gradient and breaks out of the minibatch and epoch loops when its mean exceeds target_kl.
// Here the mean is tested on the device, by the kernel that applies the update (from the per-tile
// sums that the loss gradients leave; kl_flag[0] is raised and stays raised), and that kernel
// does nothing once the flag is up: the parameters end exactly where
// the reference's break leaves them, without a host round trip.  kl_flag[2] counts the updates
// that were applied, for the host's optimiser step counters.
#include "mrl_host.hpp"
#include "mrl_device.hpp"
#include "mlp_split.hpp"
#include "mlp3.hpp"
#include "tile_sums.hpp"
#include "ppo_grads.hpp"
#include <chrono>

namespace mrl {

constexpr int UTPB = 256;

MRL_DEV float u_wave_sum(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}
template <int NW>
MRL_DEV float u_block_sum(float v, float *smem) {
    v = u_wave_sum(v);
    if ((threadIdx.x & 63) == 0) smem[threadIdx.x >> 6] = v;
    __syncthreads();
    float t = 0.0f;
#pragma unroll
    for (int k = 0; k < NW; ++k) t += smem[k];
    __syncthreads();
    return t;
}

// ppo_gather_minibatch_kernel (ppo.mojo:135-191) with the per-minibatch advantage normalisation
// (ppo.mojo:2478-2511) done by one extra workgroup: that one gathers the advantages itself and
// writes them normalised, the others copy the remaining fields.
struct GatherArgs {
    const int32_t *idx;
    const float *r_obs, *r_act, *r_adv, *r_ret, *r_logp, *r_val;
    float *mb_obs, *mb_act, *mb_adv, *mb_ret, *mb_logp, *mb_val;
    int mb, obs_dim, act_dim, normalize;
};

__global__ __launch_bounds__(UTPB) void gather_norm_kernel(GatherArgs g) {
    __shared__ float smem[4];
    if (blockIdx.x == gridDim.x - 1) {
        constexpr int PER = 32;   // minibatches up to 8192 samples stay in registers
        if (g.mb <= PER * UTPB) {
            int src[PER];
            float v[PER];
#pragma unroll
            for (int k = 0; k < PER; ++k) {
                const int i = threadIdx.x + k * UTPB;
                src[k] = i < g.mb ? g.idx[i] : -1;
            }
#pragma unroll
            for (int k = 0; k < PER; ++k) v[k] = src[k] >= 0 ? g.r_adv[src[k]] : 0.0f;
            if (g.normalize) {
                float s = 0.0f;
#pragma unroll
                for (int k = 0; k < PER; ++k) s += v[k];
                const float mean = u_block_sum<4>(s, smem) / (float)g.mb;
                float q = 0.0f;
#pragma unroll
                for (int k = 0; k < PER; ++k) {
                    const float d = v[k] - mean;
                    q += src[k] >= 0 ? d * d : 0.0f;
                }
                const float variance = u_block_sum<4>(q, smem) / (float)g.mb;
                const float std = sqrtf(variance + 1e-8f);
#pragma unroll
                for (int k = 0; k < PER; ++k) v[k] = (v[k] - mean) / (std + 1e-8f);
            }
#pragma unroll
            for (int k = 0; k < PER; ++k)
                if (src[k] >= 0) g.mb_adv[threadIdx.x + k * UTPB] = v[k];
            return;
        }
        float s = 0.0f;
        for (int i = threadIdx.x; i < g.mb; i += UTPB) s += g.r_adv[g.idx[i]];
        if (!g.normalize) {
            for (int i = threadIdx.x; i < g.mb; i += UTPB) g.mb_adv[i] = g.r_adv[g.idx[i]];
            return;
        }
        const float mean = u_block_sum<4>(s, smem) / (float)g.mb;
        float q = 0.0f;
        for (int i = threadIdx.x; i < g.mb; i += UTPB) {
            const float d = g.r_adv[g.idx[i]] - mean;
            q += d * d;
        }
        const float variance = u_block_sum<4>(q, smem) / (float)g.mb;
        const float std = sqrtf(variance + 1e-8f);
        for (int i = threadIdx.x; i < g.mb; i += UTPB) g.mb_adv[i] = (g.r_adv[g.idx[i]] - mean) / (std + 1e-8f);
        return;
    }
    const long i = (long)blockIdx.x * UTPB + threadIdx.x;
    const int w = g.obs_dim;
    if (i >= (long)g.mb * w) return;
    const int b = (int)(i / w), c = (int)(i - (long)b * w);
    const long src = g.idx[b];
    g.mb_obs[i] = g.r_obs[src * g.obs_dim + c];
    if (c < g.act_dim) g.mb_act[(long)b * g.act_dim + c] = g.r_act[src * g.act_dim + c];
    if (c == 0) {
        g.mb_ret[b] = g.r_ret[src];
        g.mb_logp[b] = g.r_logp[src];
        g.mb_val[b] = g.r_val[src];
    }
}

// Mean and standard deviation of the advantages of minibatch blockIdx.x (rows idx[k * mb ..]), with
// the arithmetic of the normalising workgroup of gather_norm_kernel: stats[2k] = mean,
// stats[2k + 1] = sqrt(variance + 1e-8).  The fused forward normalises with them on the fly.
__global__ __launch_bounds__(UTPB) void adv_stats_kernel(const int32_t *__restrict__ idx,
                                                         const float *__restrict__ r_adv, int mb,
                                                         float *__restrict__ stats) {
    __shared__ float smem[4];
    constexpr int PER = 32;
    const int32_t *my = idx + (size_t)blockIdx.x * mb;
    float mean, variance;
    if (mb <= PER * UTPB) {
        float v[PER];
        bool in[PER];
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const int i = threadIdx.x + k * UTPB;
            in[k] = i < mb;
            v[k] = in[k] ? r_adv[my[i]] : 0.0f;
        }
        float s = 0.0f;
#pragma unroll
        for (int k = 0; k < PER; ++k) s += v[k];
        mean = u_block_sum<4>(s, smem) / (float)mb;
        float q = 0.0f;
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const float d = v[k] - mean;
            q += in[k] ? d * d : 0.0f;
        }
        variance = u_block_sum<4>(q, smem) / (float)mb;
    } else {
        float s = 0.0f;
        for (int i = threadIdx.x; i < mb; i += UTPB) s += r_adv[my[i]];
        mean = u_block_sum<4>(s, smem) / (float)mb;
        float q = 0.0f;
        for (int i = threadIdx.x; i < mb; i += UTPB) {
            const float d = r_adv[my[i]] - mean;
            q += d * d;
        }
        variance = u_block_sum<4>(q, smem) / (float)mb;
    }
    if (threadIdx.x == 0) {
        stats[2 * blockIdx.x] = mean;
        stats[2 * blockIdx.x + 1] = sqrtf(variance + 1e-8f);
    }
}

// Actor and critic loss gradients in one launch (grid.y = 0: actor, 1: critic) and the KL test:
// every actor workgroup leaves the sum of its samples' KL estimates, the last one to arrive adds
// them up in workgroup order, compares the mean with target_kl and re-arms the counter.
struct LossArgs {
    const float *actor_out, *mb_logp, *mb_adv, *mb_act, *values, *mb_val, *mb_ret;
    float *g_actor_out, *g_values, *kl;
    float *kl_part;      // [grid.x]
    int *arrived;        // zero between launches
    int32_t *kl_flag;    // nullable: no test
    int mb, A, continuous, clip_value;
    float clip_eps, ent_coef, value_coef, target_kl;
};

__global__ __launch_bounds__(UTPB) void loss_grads_kernel(LossArgs a) {
    __shared__ float smem[4];
    __shared__ int last;
    const int b = blockIdx.x * UTPB + threadIdx.x;
    if (blockIdx.y == 1) {
        if (b < a.mb)
            a.g_values[b] = critic_grad_one(b, a.values, a.mb_val, a.mb_ret, a.mb, a.continuous, a.clip_value,
                                            a.value_coef, a.clip_eps);
        return;
    }
    float kl = 0.0f;
    if (b < a.mb) {
        kl = a.continuous ? actor_grad_gaussian_one(b, a.actor_out, a.mb_logp, a.mb_adv, a.mb_act, a.mb, a.A,
                                                    a.clip_eps, a.ent_coef, a.g_actor_out)
                          : actor_grad_discrete_one(b, a.actor_out, a.mb_logp, a.mb_adv, a.mb_act, a.mb, a.A,
                                                    a.clip_eps, a.ent_coef, a.g_actor_out);
        a.kl[b] = kl;
    }
    if (a.kl_flag == nullptr) return;
    const float s = u_block_sum<4>(kl, smem);
    if (threadIdx.x == 0) {
        __hip_atomic_store(&a.kl_part[blockIdx.x], s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __threadfence();
        last = atomicAdd(a.arrived, 1) == (int)gridDim.x - 1;
    }
    __syncthreads();
    if (!last) return;
    __threadfence();
    float t = 0.0f;
    for (int i = threadIdx.x; i < (int)gridDim.x; i += UTPB)
        t += __hip_atomic_load(&a.kl_part[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    t = u_block_sum<4>(t, smem);
    if (threadIdx.x == 0) {
        const float mean = t / (float)a.mb;
        a.kl_flag[1] = __float_as_int(mean);
        if (mean > a.target_kl) a.kl_flag[0] = 1;
        *a.arrived = 0;
    }
}

struct AdamNet {
    float *p, *g;
    float2 *state;
    int n;
    float lr, bc1, bc2;
    int clamp_off, clamp_n;   // log_std slice to clamp to [-5, 2] after the step (clamp_n = 0: none)
};
struct AdamNets { AdamNet n[2]; };

// partial[net][block] = sum of g^2 over the block's grid-stride slice; grid = (nb, nets)
__global__ __launch_bounds__(UTPB) void sq_partial2_kernel(AdamNets nets, float *__restrict__ partial) {
    __shared__ float smem[4];
    const AdamNet &a = nets.n[blockIdx.y];
    float s = 0.0f;
    for (long i = (long)blockIdx.x * UTPB + threadIdx.x; i < a.n; i += (long)gridDim.x * UTPB) s += a.g[i] * a.g[i];
    s = u_block_sum<4>(s, smem);
    if (threadIdx.x == 0) partial[blockIdx.y * gridDim.x + blockIdx.x] = s;
}

struct AdamArgs {
    AdamNets nets;
    const float *partial;   // sums of squares of the gradients, [net * part_stride + block], nb blocks
    int nb, part_stride;
    float max_norm, beta1, beta2, omb1, omb2, eps;
    int32_t *stop;          // the KL early stop's flag words (null: no test)
    // not null: the KL early-stop test of this minibatch has not been made yet: kl_part[0 .. kl_n) hold the row
    // tiles' sums of the per-sample estimates
    const float *kl_part;
    int kl_n, kl_mb;
    float target_kl;
    // not null: where the host looks for the stop while it enqueues a call's minibatches; gets the call's number
    int *stop_seen;
    int stop_call;
    // not null: gets the number of this minibatch, for the host to see how far the device is
    unsigned *reached, count;
};

// Whether the update is applied (it is not once stop[0] != 0), and the factor of the global-norm clip (ppo.mojo:382-534;
// actor and critic separately).  Both sums are taken side by side.  Every workgroup adds the tiles' KL sums up in the same
// order; workgroup (0, 0) records the verdict (stop[0] raised and sticky, stop[1] = the mean's bits, stop[2] counts the
// updates applied).  It does so while other workgroups still read stop[0], so the word is read once per workgroup, by
// thread 0, whose decision all wavefronts take behind the barrier: a workgroup that finds the flag raised by this very
// launch and one that does not come to the same end, the second by its own sum.  (Against every wavefront leaving as soon as
// it reads the flag: an update of 512 minibatches of 256 rows, H = 64, most of them behind the stop, 6.04 -> 6.11 ms where
// two runs of one build differ by 0.11.)
MRL_DEV bool clip_verdict(const AdamArgs &a, float *smem, float &scale) {
    __shared__ int stop_s;
    scale = 1.0f;
    const int raised = a.stop != nullptr && threadIdx.x == 0 ? a.stop[0] : 0;
    float s = 0.0f;
    if (a.max_norm > 0.0f)
        for (int i = threadIdx.x; i < a.nb; i += UTPB) s += a.partial[blockIdx.y * a.part_stride + i];
    if (a.stop != nullptr && threadIdx.x < 64) {
        float sum = 0.0f;
        if (a.kl_part != nullptr) {
            for (int i = threadIdx.x; i < a.kl_n; i += 64) sum += a.kl_part[i];
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
        }
        if (threadIdx.x == 0) {
            const float mean = sum / (float)a.kl_mb;
            const bool over = a.kl_part != nullptr && mean > a.target_kl;
            stop_s = raised != 0 || over;
            if (a.reached != nullptr && blockIdx.x == 0 && blockIdx.y == 0)
                __hip_atomic_store(a.reached, a.count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            if (stop_s && a.stop_seen != nullptr && blockIdx.x == 0 && blockIdx.y == 0)
                __hip_atomic_store(a.stop_seen, a.stop_call, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            if (a.kl_part != nullptr && raised == 0 && blockIdx.x == 0 && blockIdx.y == 0) {
                a.stop[1] = __float_as_int(mean);
                if (over) a.stop[0] = 1;
            }
        }
    }
    s = u_block_sum<4>(s, smem);
    if (a.stop != nullptr && stop_s) return false;
    if (a.max_norm > 0.0f) {
        const float norm = sqrtf(s);
        scale = norm > a.max_norm ? a.max_norm / (norm + 1e-8f) : 1.0f;
    }
    if (a.stop != nullptr && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) a.stop[2] = a.stop[2] + 1;
    return true;
}

// Adam (adam.mojo:52-105) on one parameter: gi = its clipped gradient
template <class Args>
MRL_DEV float adam_one(const Args &a, const AdamNet &net, float p, float gi, float &m, float &v) {
    m = a.beta1 * m + a.omb1 * gi;
    v = a.beta2 * v + a.omb2 * gi * gi;
    const float m_hat = m / net.bc1, v_hat = v / net.bc2;
    return p - net.lr * m_hat / (sqrtf(v_hat) + a.eps);
}

MRL_DEV float clamp_log_std(float p) { return p < -5.0f ? -5.0f : (p > 2.0f ? 2.0f : p); }

// clip + Adam + log_std clamp (kernels.mojo:842-873) of element i
MRL_DEV void adam_element(const AdamArgs &a, const AdamNet &net, int i, float p0, float g0, float2 mv, float scale) {
    const float gi = g0 * scale;
    net.g[i] = gi;
    float p = adam_one(a, net, p0, gi, mv.x, mv.y);
    net.state[i] = mv;
    if (i >= net.clamp_off && i < net.clamp_off + net.clamp_n) p = clamp_log_std(p);
    net.p[i] = p;
}

// any nets; grid = (blocks, nets)
__global__ __launch_bounds__(UTPB) void clip_adam2_kernel(AdamArgs a) {
    __shared__ float smem[4];
    const AdamNet &net = a.nets.n[blockIdx.y];
    const int i = blockIdx.x * UTPB + threadIdx.x;
    float p = 0.0f, g = 0.0f;
    float2 mv = make_float2(0.0f, 0.0f);
    if (i < net.n) { p = net.p[i]; g = net.g[i]; mv = net.state[i]; }
    float scale;
    if (!clip_verdict(a, smem, scale)) return;
    if (i < net.n) adam_element(a, net, i, p, g, mv, scale);
}

// The fused nets (hidden width H, W1 at offset o1): the first H * H / 2048 workgroups take eight consecutive columns of
// W1 per thread and keep the split operand copies of mlp_split.hpp in step (null: not kept); the others take the
// remaining parameters one per thread.  Everything that does not depend on the verdict is requested ahead of it.
// Parameters lie on 16 bytes (the row tiles need that); gradients and moments may lie on any float, for instance as slices
// of one vector: the same 16-byte accesses reach them there.
template <int H>
__global__ __launch_bounds__(UTPB) void clip_adam_split_kernel(AdamArgs a, int o1, SplitNets sp) {
    constexpr int WB = H * H / (8 * UTPB), ROWS = 8 * UTPB / H, TLD = H + 4;
    __shared__ float smem[4];
    __shared__ __align__(16) float tile[ROWS * TLD];
    const AdamNet &net = a.nets.n[blockIdx.y];
    const int t = threadIdx.x;
    float scale;
    if (blockIdx.x >= WB) {
        int i = (blockIdx.x - WB) * UTPB + t;
        if (i >= o1) i += H * H;
        float p = 0.0f, g = 0.0f;
        float2 mv = make_float2(0.0f, 0.0f);
        if (i < net.n) { p = net.p[i]; g = net.g[i]; mv = net.state[i]; }
        if (!clip_verdict(a, smem, scale)) return;
        if (i < net.n) adam_element(a, net, i, p, g, mv, scale);
        return;
    }
    const int rl = t / (H / 8), c8 = t % (H / 8), row = blockIdx.x * ROWS + rl;
    const size_t off = (size_t)o1 + (size_t)row * H + 8 * c8;
    f32x4 p[2];
    f32x4a4 g[2], st[4];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        p[k] = *reinterpret_cast<const f32x4 *>(net.p + off + 4 * k);
        g[k] = *reinterpret_cast<const f32x4a4 *>(net.g + off + 4 * k);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) st[k] = *reinterpret_cast<const f32x4a4 *>(net.state + off + 2 * k);
    if (!clip_verdict(a, smem, scale)) return;
    f32x8 pn;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const float gi = g[k >> 2][k & 3] * scale;
        g[k >> 2][k & 3] = gi;
        float m = st[k >> 1][2 * (k & 1)], v = st[k >> 1][2 * (k & 1) + 1];
        pn[k] = adam_one(a, net, p[k >> 2][k & 3], gi, m, v);
        st[k >> 1][2 * (k & 1)] = m;
        st[k >> 1][2 * (k & 1) + 1] = v;
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        *reinterpret_cast<f32x4a4 *>(net.g + off + 4 * k) = g[k];
        const f32x4 q = {pn[4 * k], pn[4 * k + 1], pn[4 * k + 2], pn[4 * k + 3]};
        *reinterpret_cast<f32x4 *>(net.p + off + 4 * k) = q;
        *reinterpret_cast<f32x4 *>(tile + rl * TLD + 8 * c8 + 4 * k) = q;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) *reinterpret_cast<f32x4a4 *>(net.state + off + 2 * k) = st[k];
    if (sp.wf[0] == nullptr) return;
    bf16x8 pc[SPLIT];
    split8(pn, pc);
    unsigned short *wb = sp.wb[blockIdx.y], *wf = sp.wf[blockIdx.y];
#pragma unroll
    for (int i = 0; i < SPLIT; ++i)
        *reinterpret_cast<bf16x8 *>(wb + split_frag<H>(c8 >> 2, row >> 4, i, (c8 & 3) * 16 + (row & 15))) = pc[i];
    __syncthreads();
    const int col = t % H, kg = t / H, k8 = blockIdx.x * (ROWS / 8) + kg;
    f32x8 x;
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = tile[(8 * kg + j) * TLD + col];
    split8(x, pc);
#pragma unroll
    for (int i = 0; i < SPLIT; ++i)
        *reinterpret_cast<bf16x8 *>(wf + split_frag<H>(k8 >> 2, col >> 4, i, (k8 & 3) * 16 + (col & 15))) = pc[i];
}

template <int H>
static void launch_adam_split(hipStream_t st, const AdamArgs &a, int o1, const SplitNets &sp) {
    const int nmax = std::max(a.nets.n[0].n, a.nets.n[1].n);
    hipLaunchKernelGGL(clip_adam_split_kernel<H>, dim3(H * H / (8 * UTPB) + grid_for(nmax - H * H, UTPB), 2), dim3(UTPB), 0,
                       st, a, o1, sp);
}

// The sums over the tiles and splits, clip and Adam in one launch (the fused nets again).  A workgroup adds up the pieces of
// its parameters, leaves the sum of their squares in `posts` for the others of its net, waits until all of these
// are there and goes on to Adam with its gradients in registers: what crosses the chip between the two is 8 bytes per workgroup,
// not the gradients, and a launch less is 2.5 us.  What bounds it: four trips to memory one after the other -- arguments,
// pieces, the squares out, the squares in (H = 64, 256 rows: 8.5 thousand cycles, of which the pieces 2.8, the exchange 3.9),
// and from H = 128 on the pieces' bytes (10 and 15 MB at 1000 and 4096 rows).  us per minibatch with sum3_kernel and
// clip_adam_split_kernel : in one launch: H = 64, 256 rows 18.0 : 14.5; H = 128, 1000 rows 27.7 : 24.9; H = 256,
// 4096 rows 55.5 : 52.7.
//
// The wait is a short one where every workgroup of the grid is on the chip, so the host takes this kernel only where the grid
// is no larger than the CUs that the stream may use.  It does not need that: other streams and processes may hold the places
// of a part of the grid for as long as they like, also with waits of their own.  After `patience` polls a workgroup adds up the
// squares that it still misses by itself, from the pieces, which nothing writes meanwhile: the same terms in the same order, so
// the same bits.  (A limit of polls below that, which only a test sets, ends the wait before: the workgroup reports it and
// updates nothing.)
// W1: VW neighbouring columns per thread, so that a workgroup holds ROWS whole rows; the rest one parameter per thread.
struct SumAdam {
    struct Net {
        AdamNet adam;
        SumNet sum;
        unsigned short *wf, *wb;   // split copies of W1; null: not kept
    } net[2];
    float max_norm, beta1, beta2, omb1, omb2, eps;
    int IN, tiles;
    const int32_t *skip;      // never null
    uint64_t *posts;          // [net][gridDim.x]: 2^32 + the bits of a workgroup's sum of squares; zero before the launch
    unsigned patience, spin_limit;
    int *sync_error;
    int32_t *stop;            // the KL early stop's flag words; without a test a place with a zero and kl_n = 0
    const float *kl_part;     // the row tiles' sums, never null
    int kl_n, kl_mb;
    float target_kl;
    int *stop_seen, stop_call;        // as in AdamArgs
    unsigned *reached, count;
};

template <int H, bool TREE>
__global__ __launch_bounds__(UTPB, 4) void sum_adam_kernel(SumAdam k) {
    constexpr int VW = H == 256 ? 4 : 1, E = UTPB * VW, ROWS = E / H, WB = H * H / E, TLD = H + 4, NW = UTPB / 64;
    constexpr int KL_MOST = 1024;     // row tiles (update_paired)
    typedef float MV __attribute__((ext_vector_type(2 * VW), aligned(4)));
    typedef float V1 __attribute__((ext_vector_type(VW), aligned(4)));
    typedef std::conditional_t<VW == 1, float, f32x4> Sum;
    __shared__ __align__(16) float tile[ROWS * TLD];
    __shared__ float sq_s[NW], kl_s[NW], total_s;
    __shared__ uint64_t word_s[64];
    __shared__ int state_s;    // 0: update, 1: the KL stop, 2: the wait gave up, 3: no longer waiting for the others' sums
    const int ynet = blockIdx.y, t = threadIdx.x;
    const SumAdam::Net net = k.net[ynet];
    const bool test = k.kl_n > 0;
    // ---- requests
    const int32_t skip = *k.skip, raised = k.stop[0];
    float klq[KL_MOST / UTPB];
#pragma unroll
    for (int j = 0; j < KL_MOST / UTPB; ++j) klq[j] = k.kl_part[max(min(t + j * UTPB, k.kl_n - 1), 0)];
    const int o1 = (k.IN + 1) * H;
    const int TB = gridDim.x - WB;                    // the thin layers' workgroups go first: theirs are the long sums
    struct Place { bool hidden, mine; int e0, i; };   // element of W1, parameter
    auto place = [&](int block) {
        Place at;
        at.hidden = block >= TB;
        at.e0 = (block - TB) * E + VW * t;
        int thin = block * UTPB + t;                  // a thin layer's parameter
        if (thin >= o1) thin += H * H;
        at.mine = at.hidden || thin < net.adam.n;
        at.i = at.hidden ? o1 + at.e0 : min(thin, net.adam.n - 1);
        return at;
    };
    auto thin_sum = [&](const Place &at) {
        const float x = sum_terms<TREE, float>(thin_terms(net.sum, k.IN, H, k.tiles, at.i));
        return at.mine ? x : 0.0f;
    };
    auto square = [](const Sum &s) {
        if constexpr (VW == 1) return s * s;
        else return (s[0] * s[0] + s[1] * s[1]) + (s[2] * s[2] + s[3] * s[3]);
    };
    const Place own_place = place(blockIdx.x);
    const bool hidden = own_place.hidden, mine = own_place.mine;
    const int i = own_place.i;
    V1 p = V1{};
    MV mv = MV{};
    Sum s = Sum{};
    if (hidden) {
        p = *reinterpret_cast<const V1 *>(net.adam.p + i);
        mv = *reinterpret_cast<const MV *>(net.adam.state + i);
        __builtin_amdgcn_sched_barrier(0);
        s = sum_terms<TREE, Sum>(hidden_terms(net.sum, own_place.e0));
    } else {
        const float2 one = net.adam.state[i];
        p[0] = net.adam.p[i];
        __builtin_amdgcn_sched_barrier(0);
        const float x = thin_sum(own_place);
        mv[0] = one.x;
        mv[1] = one.y;
        if constexpr (VW == 1) s = x;
        else s[0] = x;
    }
    // ---- the KL verdict, the same in every workgroup, and the norm
    float q = square(s), kl = 0.0f;
#pragma unroll
    for (int j = 0; j < KL_MOST / UTPB; ++j) kl += t + j * UTPB < k.kl_n ? klq[j] : 0.0f;
    q = dpp_wave_sum(q);
    kl = dpp_wave_sum(kl);
    if ((t & 63) == 0) { sq_s[t >> 6] = q; kl_s[t >> 6] = kl; }
    __syncthreads();
    uint64_t *const post = k.posts + (size_t)ynet * gridDim.x;
    auto post_word = [&](int block, float sum) {
        __hip_atomic_store(post + block, (1ull << 32) | __float_as_uint(sum), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    auto posted = [&](int block) { return __hip_atomic_load(post + block, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
    if (t < 64) {
        const float mean = ((kl_s[0] + kl_s[1]) + (kl_s[2] + kl_s[3])) / (float)k.kl_mb;
        const bool over = test && mean > k.target_kl;
        const bool first = __builtin_amdgcn_readfirstlane(raised) == 0;
        const bool stop = test && (!first || over);
        int state = stop ? 1 : 0;
        float total = 0.0f;
        if (!stop && k.max_norm > 0.0f) {
            if (t == 0) post_word(blockIdx.x, (sq_s[0] + sq_s[1]) + (sq_s[2] + sq_s[3]));
            // lane t takes the words t, t + 64, ..., one wait after the other: all but the first find theirs there
            unsigned polls = 0;
            for (int b0 = 0; b0 < (int)gridDim.x && state == 0; b0 += 64) {
                const bool in = b0 + t < (int)gridDim.x;
                uint64_t word = 0;
                for (;;) {
                    if (in && word == 0) word = posted(b0 + t);
                    if (!any_lane(in && word == 0)) break;
                    if (++polls >= k.patience) { state = 3; break; }
                    if (polls > k.spin_limit) { state = 2; break; }
                }
                total += __uint_as_float((uint32_t)word);
            }
            total = dpp_wave_sum(total);
        }
        if (t == 0) {
            total_s = total;
            state_s = state;
            if (state == 2) __hip_atomic_store(k.sync_error, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            if (k.reached != nullptr && blockIdx.x == 0 && ynet == 0)
                __hip_atomic_store(k.reached, k.count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            if (stop && k.stop_seen != nullptr && blockIdx.x == 0 && ynet == 0)
                __hip_atomic_store(k.stop_seen, k.stop_call, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            if (test && first && blockIdx.x == 0 && ynet == 0) {
                k.stop[1] = __float_as_int(mean);
                if (over) k.stop[0] = 1;
            }
        }
    }
    __syncthreads();
    if (state_s == 3) {
        // The words in the same order as above, lane t's t, t + 64, ...; one that is not there is worked out by all threads, as its
        // own workgroup does it, and left for the others.
        float total = 0.0f;
        for (int b0 = 0; b0 < (int)gridDim.x; b0 += 64) {
            const int n = min(64, (int)gridDim.x - b0);
            if (t < n) word_s[t] = posted(b0 + t);
            __syncthreads();
            for (int j = 0; j < n; ++j) {
                if (word_s[j] != 0) continue;
                const Place at = place(b0 + j);
                Sum x = Sum{};
                if (at.hidden) {
                    x = sum_terms<TREE, Sum>(hidden_terms(net.sum, at.e0));
                } else {
                    const float one = thin_sum(at);
                    if constexpr (VW == 1) x = one;
                    else x[0] = one;
                }
                const float sq = dpp_wave_sum(square(x));
                if ((t & 63) == 0) sq_s[t >> 6] = sq;
                __syncthreads();
                if (t == j) {
                    const float sum = (sq_s[0] + sq_s[1]) + (sq_s[2] + sq_s[3]);
                    post_word(b0 + j, sum);
                    word_s[j] = __float_as_uint(sum);
                }
                __syncthreads();
            }
            if (t < n) total += __uint_as_float((uint32_t)word_s[t]);
            __syncthreads();
        }
        if (t < 64) {
            total = dpp_wave_sum(total);
            if (t == 0) total_s = total;
        }
        __syncthreads();
    }
    const int state = state_s;
    if (state == 1 || state == 2) {
        // The gradients as they are.  (Nothing else hangs on `skip`: a workgroup of this launch may raise it while a wavefront
        // reads it.)
        if (state == 1 && skip == 0) {
            if (hidden) *reinterpret_cast<V1 *>(net.adam.g + i) = s;
            else if (mine) {
                if constexpr (VW == 1) net.adam.g[i] = s;
                else net.adam.g[i] = s[0];
            }
        }
        return;
    }
    float scale = 1.0f;
    if (k.max_norm > 0.0f) {
        const float norm = sqrtf(total_s);
        scale = norm > k.max_norm ? k.max_norm / (norm + 1e-8f) : 1.0f;
    }
    if (test && blockIdx.x == 0 && ynet == 0 && t == 0) k.stop[2] = k.stop[2] + 1;
    V1 g = V1{};
#pragma unroll
    for (int j = 0; j < VW; ++j) {
        if constexpr (VW == 1) g[j] = s * scale;
        else g[j] = s[j] * scale;
        if (j > 0 && !hidden) continue;
        float m = mv[2 * j], v = mv[2 * j + 1];
        p[j] = adam_one(k, net.adam, p[j], g[j], m, v);
        mv[2 * j] = m;
        mv[2 * j + 1] = v;
    }
    if (!hidden) {
        if (!mine) return;
        const bool clamped = i >= net.adam.clamp_off && i < net.adam.clamp_off + net.adam.clamp_n;
        net.adam.g[i] = g[0];
        net.adam.state[i] = make_float2(mv[0], mv[1]);
        net.adam.p[i] = clamped ? clamp_log_std(p[0]) : p[0];
        return;
    }
    *reinterpret_cast<V1 *>(net.adam.g + i) = g;
    *reinterpret_cast<V1 *>(net.adam.p + i) = p;
    *reinterpret_cast<MV *>(net.adam.state + i) = mv;
    if (net.wf == nullptr) return;
    // ---- the split copies: eight columns of a row, ROWS rows of a column
    const int row0 = ((int)blockIdx.x - TB) * ROWS;
#pragma unroll
    for (int j = 0; j < VW; ++j) tile[(VW * t) / H * TLD + (VW * t) % H + j] = p[j];
    __syncthreads();
    if (t < E / 8) {
        const int c8 = t % (H / 8), rl = t / (H / 8), row = row0 + rl;
        f32x8 x;
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = tile[rl * TLD + 8 * c8 + j];
        bf16x8 pc[SPLIT];
        split8(x, pc);
#pragma unroll
        for (int j = 0; j < SPLIT; ++j)
            *reinterpret_cast<bf16x8 *>(net.wb + split_frag<H>(c8 >> 2, row >> 4, j, (c8 & 3) * 16 + (row & 15))) = pc[j];
    }
    const int col = t - (UTPB - H);     // (at small widths the last wavefronts)
    if (col >= 0) {
        typedef float FR __attribute__((ext_vector_type(ROWS)));
        typedef __bf16 BR __attribute__((ext_vector_type(ROWS)));
        FR x;
#pragma unroll
        for (int j = 0; j < ROWS; ++j) x[j] = tile[j * TLD + col];
        BR pc[SPLIT];
        split_n<ROWS>(x, pc);
        const int k8 = row0 >> 3;
#pragma unroll
        for (int j = 0; j < SPLIT; ++j)
            *reinterpret_cast<BR *>(net.wf + split_frag<H>(k8 >> 2, col >> 4, j, (k8 & 3) * 16 + (col & 15)) + (row0 & 7)) = pc[j];
    }
}

static int sum_adam_blocks(int H, const AdamArgs &a) {   // per net
    return H * H / (UTPB * (H == 256 ? 4 : 1)) + grid_for(std::max(a.nets.n[0].n, a.nets.n[1].n) - H * H, UTPB);
}
template <int H>
static void launch_sum_adam(hipStream_t st, const SumAdam &k, int blocks, bool tree) {
    const dim3 grid(blocks, 2);
    if (tree) hipLaunchKernelGGL((sum_adam_kernel<H, true>), grid, dim3(UTPB), 0, st, k);
    else hipLaunchKernelGGL((sum_adam_kernel<H, false>), grid, dim3(UTPB), 0, st, k);
}

}  // namespace mrl

using namespace mrl;

extern "C" {

static int update_check(const mrl_update *u, const char *who) {
    MRL_CHECK_ARG(u != nullptr, "%s: descriptor is NULL", who);
    MRL_CHECK_ARG(u->minibatch > 0 && u->obs_dim > 0 && u->act_width > 0, "%s: bad sizes", who);
    MRL_CHECK_ARG(u->actor_params && u->critic_params && u->actor_grads && u->critic_grads && u->actor_state &&
                      u->critic_state, "%s: NULL parameter / gradient / optimiser buffer", who);
    MRL_CHECK_ARG(u->r_obs && u->r_actions && u->r_log_probs && u->r_values && u->advantages && u->returns,
                  "%s: NULL rollout buffer", who);
    MRL_CHECK_ARG(u->mb_obs && u->mb_actions && u->mb_adv && u->mb_ret && u->mb_logp && u->mb_val &&
                      u->actor_out && u->values && u->g_actor_out && u->g_values && u->kl && u->actor_cache &&
                      u->critic_cache, "%s: NULL minibatch buffer", who);
    MRL_CHECK_ARG(u->target_kl <= 0.0f || u->kl_flag != nullptr, "%s: target_kl needs kl_flag", who);
    const int head = mrl_mlp_out_dim(&u->actor);
    MRL_CHECK_ARG(head > 0 && mrl_mlp_out_dim(&u->critic) == 1, "%s: bad actor / critic description", who);
    const bool gauss = u->actor.layers[u->actor.n_layers - 1].kind == MRL_STOCHASTIC_ACTOR;
    MRL_CHECK_ARG(gauss == (u->continuous != 0), "%s: a continuous agent needs a StochasticActor head (and only it)",
                  who);
    MRL_CHECK_ARG(!gauss || head == 2 * u->act_width, "%s: act_width does not match the actor head", who);
    MRL_CHECK_ARG(gauss || u->act_width == 1, "%s: a discrete agent stores one float per action", who);
    MRL_CHECK_ARG(u->actor.layers[0].in_dim == u->obs_dim && u->critic.layers[0].in_dim == u->obs_dim,
                  "%s: nets do not read obs_dim inputs", who);
    return MRL_OK;
}

// floats of ctx->upd_scratch: KL partials, their arrival counter, sum-of-squares partials, and the
// advantage statistics of up to STATS_MAX minibatches
constexpr int SCR_KL = 0, SCR_ARRIVED = 1024, SCR_SQ = 2048, SCR_STATS = 4096, STATS_MAX = 2048;
constexpr int POSTS_MAX = 1024;   // 8-byte words of sum_adam_kernel where the sum-of-squares partials lie otherwise

// both nets of the fused shapes, parameters that 16-byte loads can reach, a KL sum per row tile
static bool update_paired(const mrl_update *u) {
    return mlp3_pair_fusable(u->actor, u->critic) && reinterpret_cast<uintptr_t>(u->actor_params) % 16 == 0 &&
           reinterpret_cast<uintptr_t>(u->critic_params) % 16 == 0 && (u->minibatch + 31) / 32 <= 1024;
}

static void adam_args(const mrl_update *u, int actor_t, int critic_t, AdamArgs &a) {
    const int Pa = mrl_mlp_param_size(&u->actor), Pc = mrl_mlp_param_size(&u->critic);
    auto fill = [&](AdamNet &n, float *p, float *g, float *st, int size, double lr, int t) {
        n.p = p; n.g = g; n.state = reinterpret_cast<float2 *>(st); n.n = size; n.lr = (float)lr;
        // bias corrections in fp64 then rounded, as the host code of the reference does
        n.bc1 = (float)(1.0 - pow(u->beta1, (double)t));
        n.bc2 = (float)(1.0 - pow(u->beta2, (double)t));
        n.clamp_off = 0; n.clamp_n = 0;
    };
    fill(a.nets.n[0], u->actor_params, u->actor_grads, u->actor_state, Pa, u->actor_lr, actor_t);
    fill(a.nets.n[1], u->critic_params, u->critic_grads, u->critic_state, Pc, u->critic_lr, critic_t);
    if (u->continuous) { a.nets.n[0].clamp_off = Pa - u->act_width; a.nets.n[0].clamp_n = u->act_width; }
    a.max_norm = u->max_grad_norm;
    a.beta1 = (float)u->beta1; a.beta2 = (float)u->beta2;
    a.omb1 = (float)(1.0 - u->beta1); a.omb2 = (float)(1.0 - u->beta2); a.eps = (float)u->eps;
    a.stop = u->target_kl > 0.0f ? u->kl_flag : nullptr;
    a.kl_mb = u->minibatch;
    a.target_kl = u->target_kl;
}

// One minibatch of the fused nets; stats: {mean, std} of its advantages on the device (null: not normalised).
// ws.split holds the hidden layers' current weights; more: another minibatch of the same call follows.  Then the copies
// are kept in step with the updated weights, and once the KL stop is up nothing is computed: no parameter moves any more,
// and what else the call leaves (gradients, outputs, KL estimates) is its last minibatch's, which is always computed.
// watched: the host looks how far the device is.
static int update_minibatch_paired(mrl_ctx *ctx, const mrl_update *u, const int32_t *indices, int actor_t, int critic_t,
                                   const float *stats, const UpdateWs &ws, bool more, bool watched) {
    const bool cont = u->continuous != 0;
    const int mb = u->minibatch, head = mrl_mlp_out_dim(&u->actor);
    const mrl_mlp_desc *descs[2] = {&u->actor, &u->critic};
    Mlp3Nets io{};
    io.n[0].params = u->actor_params; io.n[0].out = u->actor_out;
    io.n[1].params = u->critic_params; io.n[1].out = u->values;
    FwdLoss fl{};
    fl.idx = indices;
    fl.r_obs = u->r_obs; fl.r_act = u->r_actions; fl.r_adv = u->advantages; fl.r_ret = u->returns;
    fl.r_logp = u->r_log_probs; fl.r_val = u->r_values;
    fl.adv_stats = u->norm_adv_per_minibatch ? stats : nullptr;
    fl.g_actor_out = u->g_actor_out; fl.g_values = u->g_values; fl.kl = u->kl;
    fl.kl_part = ctx->upd_scratch + SCR_KL;
    fl.kl_flag = u->target_kl > 0.0f ? u->kl_flag : nullptr;
    fl.skip = more && fl.kl_flag != nullptr ? fl.kl_flag : never_skip(ctx);
    fl.mb = mb; fl.A = cont ? u->act_width : head; fl.continuous = cont ? 1 : 0;
    fl.clip_value = u->clip_value ? 1 : 0;
    fl.clip_eps = u->clip_epsilon; fl.ent_coef = u->entropy_coef; fl.value_coef = u->value_loss_coef;
    AdamArgs a{};
    adam_args(u, actor_t, critic_t, a);
    a.kl_part = u->target_kl > 0.0f ? ctx->upd_scratch + SCR_KL : nullptr;
    a.kl_n = ws.tiles;
    a.stop_seen = more && a.stop != nullptr ? ctx->stop_seen : nullptr;
    a.stop_call = ctx->stop_call;
    if (watched) {
        a.reached = ctx->upd_reached;
        a.count = ++ctx->upd_count;
    }
    const int H = u->actor.layers[0].out_dim, o1 = (u->obs_dim + 1) * H;
    const int blocks = sum_adam_blocks(H, a);
    const bool one_launch = 2 * blocks <= std::min(ctx->stream_cus, POSTS_MAX);
    ctx->upd_end_launches = one_launch ? 1 : 2;
    if (one_launch) {
        fl.posts = reinterpret_cast<uint64_t *>(ctx->upd_scratch + SCR_SQ);
        fl.n_posts = 2 * blocks;
    }
    int rc = mlp3_update_n(ctx, descs, mb, io, ws, fl);
    if (rc) return rc;
    float *grads[2] = {u->actor_grads, u->critic_grads};
    const SumNets sn = mlp3_sum_nets(descs, 2, ws, grads, fl.skip);
    if (one_launch) {
        SumAdam k{};
        for (int i = 0; i < 2; ++i)
            k.net[i] = {a.nets.n[i], sn.net[i], more ? ws.split.wf[i] : nullptr, more ? ws.split.wb[i] : nullptr};
        k.max_norm = a.max_norm;
        k.beta1 = a.beta1; k.beta2 = a.beta2; k.omb1 = a.omb1; k.omb2 = a.omb2; k.eps = a.eps;
        k.IN = sn.IN; k.tiles = sn.tiles; k.skip = sn.skip;
        k.posts = fl.posts;
        k.patience = ctx->update_patience;
        k.spin_limit = ctx->spin_limit;
        k.sync_error = ctx->sync_error;
        const bool test = a.stop != nullptr;
        k.stop = test ? a.stop : const_cast<int32_t *>(never_skip(ctx));
        k.kl_part = ctx->upd_scratch + SCR_KL;
        k.kl_n = test ? ws.tiles : 0;
        k.kl_mb = mb;
        k.target_kl = a.target_kl;
        k.stop_seen = a.stop_seen;
        k.stop_call = a.stop_call;
        k.reached = a.reached;
        k.count = a.count;
        if (H == 256) launch_sum_adam<256>(ctx->stream, k, blocks, ws.rows == 16);
        else if (H == 128) launch_sum_adam<128>(ctx->stream, k, blocks, ws.rows == 16);
        else launch_sum_adam<64>(ctx->stream, k, blocks, ws.rows == 16);
        MRL_CHECK_LAUNCH();
        return MRL_OK;
    }
    SplitNets sp{};
    if (more) sp = ws.split;
    int sq_blocks = 0;   // > 0: the sums over the tiles already left the sum-of-squares partials
    rc = mlp3_sum_tiles(ctx, sn, ws.rows, u->max_grad_norm > 0.0f ? ctx->upd_scratch + SCR_SQ : nullptr, &sq_blocks);
    if (rc) return rc;
    a.partial = ctx->upd_scratch + SCR_SQ;
    a.nb = sq_blocks;
    a.part_stride = 1024;
    if (H == 256) launch_adam_split<256>(ctx->stream, a, o1, sp);
    else if (H == 128) launch_adam_split<128>(ctx->stream, a, o1, sp);
    else launch_adam_split<64>(ctx->stream, a, o1, sp);
    MRL_CHECK_LAUNCH();
    return MRL_OK;
}

// One minibatch of any other nets, layer by layer.
static int update_minibatch_layers(mrl_ctx *ctx, const mrl_update *u, const int32_t *indices, int actor_t, int critic_t) {
    int rc;
    const int mb = u->minibatch, head = mrl_mlp_out_dim(&u->actor);
    const bool cont = u->continuous != 0;
    GatherArgs g{indices, u->r_obs, u->r_actions, u->advantages, u->returns, u->r_log_probs, u->r_values,
                 u->mb_obs, u->mb_actions, u->mb_adv, u->mb_ret, u->mb_logp, u->mb_val,
                 mb, u->obs_dim, u->act_width, u->norm_adv_per_minibatch};
    MRL_CHECK_ARG(u->act_width <= u->obs_dim, "mrl_ppo_update_minibatch: action wider than observation");
    hipLaunchKernelGGL(gather_norm_kernel, dim3(grid_for((long)mb * u->obs_dim, UTPB) + 1), dim3(UTPB), 0,
                       ctx->stream, g);
    MRL_CHECK_LAUNCH();
    rc = mrl_mlp_forward(ctx, &u->actor, mb, u->mb_obs, u->actor_params, u->actor_out, u->actor_cache);
    if (rc) return rc;
    rc = mrl_mlp_forward(ctx, &u->critic, mb, u->mb_obs, u->critic_params, u->values, u->critic_cache);
    if (rc) return rc;
    const int nblk = grid_for(mb, UTPB);
    const bool test = u->target_kl > 0.0f && nblk <= 1024;
    LossArgs l{u->actor_out, u->mb_logp, u->mb_adv, u->mb_actions, u->values, u->mb_val, u->mb_ret,
               u->g_actor_out, u->g_values, u->kl, ctx->upd_scratch + SCR_KL,
               reinterpret_cast<int *>(ctx->upd_scratch + SCR_ARRIVED), test ? u->kl_flag : nullptr,
               mb, cont ? u->act_width : head, cont ? 1 : 0, u->clip_value ? 1 : 0,
               u->clip_epsilon, u->entropy_coef, u->value_loss_coef, u->target_kl};
    hipLaunchKernelGGL(loss_grads_kernel, dim3(nblk, 2), dim3(UTPB), 0, ctx->stream, l);
    MRL_CHECK_LAUNCH();
    if (u->target_kl > 0.0f && !test) {
        rc = mrl_kl_check(ctx, u->kl, mb, u->target_kl, u->kl_flag);
        if (rc) return rc;
    }
    rc = mrl_mlp_backward(ctx, &u->actor, mb, u->g_actor_out, u->actor_params, u->actor_cache, u->actor_grads,
                          nullptr);
    if (rc) return rc;
    rc = mrl_mlp_backward(ctx, &u->critic, mb, u->g_values, u->critic_params, u->critic_cache, u->critic_grads,
                          nullptr);
    if (rc) return rc;
    AdamArgs a{};
    adam_args(u, actor_t, critic_t, a);
    const int nmax = std::max(a.nets.n[0].n, a.nets.n[1].n);
    if (u->max_grad_norm > 0.0f) {
        float *part = ctx->reduce_scratch + 1024;   // [2][nb], nb <= 256
        a.nb = std::min(256, grid_for(nmax, UTPB));
        a.part_stride = a.nb;
        a.partial = part;
        hipLaunchKernelGGL(sq_partial2_kernel, dim3(a.nb, 2), dim3(UTPB), 0, ctx->stream, a.nets, part);
    }
    hipLaunchKernelGGL(clip_adam2_kernel, dim3(grid_for(nmax, UTPB), 2), dim3(UTPB), 0, ctx->stream, a);
    MRL_CHECK_LAUNCH();
    return MRL_OK;
}

constexpr auto AHEAD_PATIENCE = std::chrono::milliseconds(50);

// Minibatches 0 .. n - 1 of `indices`, with step counts t0 + 1 ..; ahead > 0: the caller waits for the end anyway, and with a
// KL test the host stays within that many minibatches of the device
static int update_minibatches(mrl_ctx *ctx, const mrl_update *u, const int32_t *indices, int n, int actor_t0, int critic_t0, int ahead) {
    int rc;
    ctx->upd_enqueued = ctx->upd_end_launches = 0;
    if (!update_paired(u)) {
        for (int k = 0; k < n; ++k) {
            rc = update_minibatch_layers(ctx, u, indices + (size_t)k * u->minibatch, actor_t0 + k + 1, critic_t0 + k + 1);
            if (rc) return rc;
            ctx->upd_enqueued += 1;
        }
        return MRL_OK;
    }
    // the split copies of the hidden layers' weights are made here, from the parameters as the caller left them, and
    // kept in step by the Adam kernel between this call's minibatches
    const mrl_mlp_desc *descs[2] = {&u->actor, &u->critic};
    const float *params[2] = {u->actor_params, u->critic_params};
    UpdateWs ws;
    rc = mlp3_update_ws(ctx, descs, 2, u->minibatch, params, &ws);
    if (rc) return rc;
    rc = launch_split_weights(ctx, u->actor.layers[0].out_dim, ws.split, 2);
    if (rc) return rc;
    // Behind the KL stop every launch ends at once, but a launch is 2.5 us of the device and up to 4 of the host.  So the host
    // looks whether the device has reported the stop for this call's number, and then goes on with
    // the last minibatch (which is always computed); and it may stay within `ahead` minibatches of the device, because what it has
    // enqueued beyond the stop runs.  Where the device does not come on for AHEAD_PATIENCE, for whatever reason, the host
    // stops waiting for the rest of the call.  A capture records all of them: nothing runs meanwhile, and a number is
    // never used again.  CartPole, 1024 envs x 128 steps, H = 64, 512 minibatches of 256 rows an epoch of which
    // the stop leaves a few dozen, us per train_gpu: 4900 when all were launched, 1105 without the limit, 878 with it.
    ctx->stop_call += 1;
    const volatile int *seen = ctx->stop_seen;
    const volatile unsigned *reached = ctx->upd_reached;
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    bool watched = u->target_kl > 0.0f && ahead > 0 && n > ahead;
    if (watched && hipStreamIsCapturing(ctx->stream, &capturing) != hipSuccess) {
        (void)hipGetLastError();
        watched = false;
    }
    watched = watched && capturing == hipStreamCaptureStatusNone;
    bool patient = watched;
    float *stats = ctx->upd_scratch + SCR_STATS;
    int have_stats = -1;   // the first of the STATS_MAX minibatches whose advantage statistics are there
    for (int k = 0; k < n; ++k) {
        if (patient && k >= ahead) {
            const auto since = std::chrono::steady_clock::now();
            while (ctx->upd_count - *reached >= (unsigned)ahead && *seen != ctx->stop_call && patient)
                patient = std::chrono::steady_clock::now() - since < AHEAD_PATIENCE;
        }
        if (u->target_kl > 0.0f && *seen == ctx->stop_call) k = n - 1;
        const int s0 = k / STATS_MAX * STATS_MAX;
        if (u->norm_adv_per_minibatch && s0 != have_stats) {   // of many minibatches in one launch
            hipLaunchKernelGGL(adv_stats_kernel, dim3(std::min(STATS_MAX, n - s0)), dim3(UTPB), 0, ctx->stream,
                               indices + (size_t)s0 * u->minibatch, u->advantages, u->minibatch, stats);
            MRL_CHECK_LAUNCH();
            have_stats = s0;
        }
        rc = update_minibatch_paired(ctx, u, indices + (size_t)k * u->minibatch, actor_t0 + k + 1, critic_t0 + k + 1,
                                     stats + 2 * (k - s0), ws, k + 1 < n, watched);
        if (rc) return rc;
        ctx->upd_enqueued += 1;
    }
    return MRL_OK;
}

int mrl_ppo_update_minibatch(mrl_ctx *ctx, const mrl_update *u, const int32_t *indices, int actor_t,
                             int critic_t) {
    MRL_CHECK_ARG(ctx != nullptr, "mrl_ppo_update_minibatch: ctx is NULL");
    int rc = update_check(u, "mrl_ppo_update_minibatch");
    if (rc) return rc;
    MRL_CHECK_ARG(indices != nullptr && actor_t >= 1 && critic_t >= 1,
                  "mrl_ppo_update_minibatch: need indices and step counts >= 1");
    return update_minibatches(ctx, u, indices, 1, actor_t - 1, critic_t - 1, 0);
}

int mrl_minibatch_adv_stats(mrl_ctx *ctx, const int32_t *indices, const float *advantages, int minibatch,
                            int n_minibatches, float *stats) {
    MRL_CHECK_ARG(ctx != nullptr, "mrl_minibatch_adv_stats: ctx is NULL");
    MRL_CHECK_ARG(minibatch > 0 && n_minibatches >= 0, "mrl_minibatch_adv_stats: bad sizes");
    if (n_minibatches == 0) return MRL_OK;
    MRL_CHECK_ARG(indices && advantages && stats, "mrl_minibatch_adv_stats: NULL buffer");
    // the launch mrl_ppo_update_epoch makes ahead of its minibatches, into the caller's buffer
    hipLaunchKernelGGL(adv_stats_kernel, dim3(n_minibatches), dim3(UTPB), 0, ctx->stream, indices, advantages,
                       minibatch, stats);
    MRL_CHECK_LAUNCH();
    return MRL_OK;
}

static int update_epoch(mrl_ctx *ctx, const mrl_update *u, const int32_t *indices, int n_minibatches, int actor_t0, int critic_t0,
                        int ahead, const char *who) {
    MRL_CHECK_ARG(ctx != nullptr, "%s: ctx is NULL", who);
    ctx->upd_enqueued = ctx->upd_end_launches = 0;
    int rc = update_check(u, who);
    if (rc) return rc;
    MRL_CHECK_ARG(n_minibatches >= 0 && actor_t0 >= 0 && critic_t0 >= 0, "%s: negative count", who);
    MRL_CHECK_ARG(n_minibatches == 0 || indices != nullptr, "%s: indices is NULL", who);
    return n_minibatches == 0 ? MRL_OK : update_minibatches(ctx, u, indices, n_minibatches, actor_t0, critic_t0, ahead);
}

int mrl_ppo_update_epoch(mrl_ctx *ctx, const mrl_update *u, const int32_t *indices, int n_minibatches,
                         int actor_t0, int critic_t0) {
    return update_epoch(ctx, u, indices, n_minibatches, actor_t0, critic_t0, 0, "mrl_ppo_update_epoch");
}

int mrl_ppo_update_epoch_ahead(mrl_ctx *ctx, const mrl_update *u, const int32_t *indices, int n_minibatches,
                               int actor_t0, int critic_t0, int ahead) {
    MRL_CHECK_ARG(ahead >= 1, "mrl_ppo_update_epoch_ahead: ahead must be positive");
    return update_epoch(ctx, u, indices, n_minibatches, actor_t0, critic_t0, ahead, "mrl_ppo_update_epoch_ahead");
}

}  // extern "C"
