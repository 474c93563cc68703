// Fused collection kernels with 16 envs per workgroup for LunarLander (both action spaces), CartPole and Pendulum,
// at hidden widths 64, 128 and 256: many rollout steps of a block's envs in one launch, as in mrl_collect.hip.
#pragma once
#include <type_traits>
#include "mrl_host.hpp"
#include "mrl_device.hpp"
#include "mlp_tile.hpp"
#include "mlp_tile16.hpp"
#include "policy_sample.hpp"
#include "env_block.hpp"
#include "env_classic.hpp"
#include "collect_args.hpp"

namespace mrl {

template <int A, int B>
constexpr int cmax() { return A > B ? A : B; }

// column tiles of 16 of the critic on the three helpers: helper 0, which draws the action once more, never more than the
// others
template <int H>
struct Critic16Split {
    static constexpr int TILES = H / 16;
    static constexpr int N0 = TILES / 3, N1 = (TILES - N0 + 1) / 2, N2 = TILES - N0 - N1;
};

// ---------------------------------------------------------------- 16 rows per workgroup
// A workgroup of four wavefronts and 16 envs.  A step is a chain -- actor on the matrix cores, then sampling and the env
// step on ONE wavefront's vector unit --, and beside it the critic, whose value is only stored.
//   all four wavefronts     actor  OBS -> H -> H -> A, 64 columns each;
//   the solver wavefront    sampling (four lanes per env), two of the fourteen detection tasks, env step (four lanes per
//                           env, one per body: env_lunar.hpp), accounting, resets;
//   the other three         contact detection, what the engines need whatever the action is, the action's log-probability,
//                           then the critic (H = 256: 80 / 96 / 80 columns) at a barrier of their own.
// Two such workgroups fit a CU (LDS, registers).  On this hardware a SIMD issues either a matrix or a vector instruction,
// never both at once (a wavefront of dependent v_fma_f32 that shares its SIMD with a wavefront issuing v_mfma back to back
// takes the sum of both times), so at H = 256 the second one costs what its forward passes cost (4096 : 8192 envs 18.5 :
// 27.3 us per step); still, since the solver carries four lanes per env, two of 16 rows are ahead of one of 32 rows with one
// lane per env and the critic on six wavefronts (33.0).
// One lane per env : four, us per step: 777 envs, H = 64 19.4 : 12.9 (its solver wavefront: 22 of 37 thousand cycles in the
// physics before); 4096 envs, H = 64 18.8 : 12.6, H = 256, where the critic is the longer path, 23.9 : 21.6.  The engines'
// sines and the log-probability off the solver, its detection in one pass of all four wavefronts: H = 64, 777 envs
// 11.46 : 11.26, 4096 envs 11.86 : 11.55 (11.2 since a step's first loads are no longer waited for; thousand cycles of a
// step there: actor 5.0, sample 1.1, detection 3.5, wait 0.8, engines 1.6, physics and tail 12, reset 1).
// The solver wavefront is 0 in the lower half of the grid and 2 in the upper half: workgroups i and
// i + grid / 2 share a CU when the grid is twice the CU count, and their solvers then sit on
// different SIMDs.
template <class E, int H, int ACT, bool GAUSS>
__global__ __launch_bounds__(256, 2) void collect16_kernel(CollectArgs a) {
    using S = Stage<E>;
    constexpr int IN = E::OBS, AW = E::ACT_W, R = PR16, T = E::THREADS;
    constexpr int NTA = H / 64;   // actor: column tiles per wavefront
    constexpr Critic16Split<H> CS{};
    constexpr int CAP = 3;      // records per (body, vertex) list: two contacts, the third signals overflow
    constexpr int KBA = 8;      // k-steps of layer-1 weights fetched ahead
    static_assert(IN <= PIN_MAX && AW <= PA_MAX && E::DETECT_TASKS >= 12 && E::DETECT_TASKS <= 16, "tile limits; split-off detection");
    __shared__ float rows[R * S::STRIDE];
    __shared__ float xs[R * XS_LD];
    __shared__ __align__(16) float w2a[HEAD_LDS(H)];
    __shared__ float w2c[H + 1];                    // the critic's head: column of H weights, then the bias
    __shared__ float logits[R * (PA_MAX + 1)];
    __shared__ float vals[R];
    __shared__ float act[R * PA_MAX];
    __shared__ float shapes[E::NSHAPE];
    __shared__ ll::EngineDraw draws[R];
    __shared__ unsigned long long was_reset;
    __shared__ unsigned sync_critic, sync_detect, sync_failed;
    __shared__ float hTc[H * HT16_LD];              // the critic's activation tile (live during the env step)
    // the actor's activation tile and the env step's contact scratch are never live together
    constexpr int LIST_F = detect_list_floats<E, CAP>() + 1;
    constexpr int ENV_F = R * S::CSTRIDE + LIST_F + detect_count_ints<E>();
    __shared__ float overlay[cmax<H * HT16_LD, ENV_F>()];
    float *cts = overlay, *dlist = cts + R * S::CSTRIDE;
    int *dcount = reinterpret_cast<int *>(dlist + LIST_F);

    const int t = threadIdx.x;
    const int env0 = blockIdx.x * R;
    const int nenv = min(R, a.n_envs - env0);
    const int N = a.n_envs;
    const int sw = (2 * blockIdx.x >= gridDim.x && gridDim.x > 1) ? 2 : 0;   // the solver wavefront
    float *gbase = a.states + (size_t)env0 * E::STATE;

    S::in(rows, gbase, nenv, t);
    for (int i = t; i < E::NSHAPE; i += T) shapes[i] = a.shapes[i];
    stage_head(a.actor_p + IN * H + H + H * H + H, H, a.A, GAUSS, w2a, t, T);
    for (int i = t; i < H + 1; i += T) w2c[i] = a.critic_p[IN * H + H + H * H + H + i];
    if (t == 0) {
        was_reset = 0;
        sync_critic = 0;
        sync_detect = 0;
        sync_failed = 0;
    }
    __syncthreads();
    // solver wavefront, four lanes per env: the env's running episode return and length stay in registers of the first,
    // and what its wiring is (E::lanes_wired) in all four
    const int my_env = (t & 63) >> 2;
    const bool owner = (t >> 6) == sw && my_env < nenv && (t & 3) == 0;
    float ep_return = owner ? a.acc.ep_return[env0 + my_env] : 0.0f;
    float ep_length = owner ? a.acc.ep_length[env0 + my_env] : 0.0f;
    int wired = my_env < nenv ? E::lanes_wired(rows + my_env * S::STRIDE) : 0;

    for (int k = 0; k < a.n_steps; ++k) {
        // Nothing but the rows is carried from one step to the next: the thread index, the block's
        // env count and the parameter pointers pass through empty asm statements at the top of each
        // step, so the optimiser cannot keep what it derives from them live through the env step,
        // whose solver needs the registers.
        int tid = t, ne = __builtin_amdgcn_readfirstlane(nenv), A = __builtin_amdgcn_readfirstlane(a.A), zero = 0;
        asm volatile("" : "+v"(tid), "+s"(zero), "+s"(ne), "+s"(A) : : "memory");
        const float *pa = a.actor_p + zero, *pc = a.critic_p + zero;
        const size_t row = (size_t)(a.t0 + k) * N + env0;   // this block's slice of rollout row t
        const uint32_t sseed = a.sample_seed + (uint32_t)k * a.sample_stride;
        const int wave = tid / WAVE, lane = tid % WAVE;
        const int vw = (wave - sw) & 3;                     // 0: solver, 1 .. 3: helpers
        // the helpers' barriers, rebuilt every step from the step number (the critic's hidden stack meets
        // three times per step, the detection once): nothing of them stays in registers through the env step
        WaveGroupSync critic_sync{&sync_critic, (unsigned)k * 9u, 3u, &sync_failed, a.spin_limit};
        WaveGroupSync detect_sync{&sync_detect, (unsigned)k * 3u, 3u, &sync_failed, a.spin_limit};
        // ---- actor, all wavefronts
        {
            Hidden16Operands<H, IN, NTA, KBA> ops;
            ops.load(pa, 16 * NTA * wave, lane);
            stage_observations<IN, T>(xs, a.r_obs + row * IN, ne, tid, [&](int r, int c) { return rows[r * S::STRIDE + c]; });
            __syncthreads();
            BlockSync bs;
            hidden_stack16<H, IN, ACT, NTA, KBA, true>(pa, xs, overlay, overlay, ops, 16 * NTA * wave, lane, bs);
            head16<H>(w2a, A, overlay, logits, PA_MAX + 1, tid, T);
            __syncthreads();   // logits complete; the actor's tile is dead from here on
        }
        if (vw == 0) {   // ---- sample
            const int e = lane >> 2;
            const bool first = (lane & 3) == 0;
            if (e < ne) {
                const int i = env0 + e;
                const float *lg = logits + e * (PA_MAX + 1);
                if (GAUSS) {
                    for (int j = lane & 3; j < A; j += 4) {   // (one component a lane)
                        float av;
                        sample_gaussian_part(lg + j, w2a + HEAD_LOG_STD(H) + j, 1, A, j, sseed, i, &av);
                        act[e * AW + j] = av;
                    }
                } else {   // (four actions: the entry refuses any other head)
                    const int sel = sample_categorical_quad(lg, A, sseed, i, lane & 3);
                    if (first) act[e] = (float)sel;
                }
            }
        } else if (vw == 3 && lane < ne) {   // ---- what the engines need whatever the action is
            draws[lane] = ll::engine_draw(rows + lane * S::STRIDE, env0 + lane);
        }
        {   // ---- contact detection: a (body, vertex) task of env slot lane % 16 each, four a helper, the solver the rest
            const int task = (vw == 0 ? 12 : 4 * (vw - 1)) + lane / R, e = lane % R;
            if (task < E::DETECT_TASKS && e < ne) detect_vertex_task<E, CAP>(rows, shapes, dlist, dcount, task, e);
        }
        if (vw == 0) {
            // ---- the env step of env_block.hpp with the contacts detected
            typename E::Carry carry{};
            const int e = lane >> 2;
            const bool first = (lane & 3) == 0 && e < ne;
            detect_sync.target += detect_sync.nwaves;
            detect_sync.wait_for(detect_sync.target);
            if (first) carry = E::step_begin(rows + e * S::STRIDE, env0 + e, act + e * AW, shapes, draws + e);
            float r = 0.0f, d = 0.0f;
            step_finish_quads<E, CAP>(rows, cts, shapes, dlist, dcount, carry, wired, lane, ne, r, d);
            bool finished = false;
            if (first) {
                a.r_rewards[row + e] = r;
                a.r_dones[row + e] = d;
                ep_return = ep_return + r;
                ep_length = ep_length + 1.0f;
                finished = d > 0.5f;
                if (finished) {
                    const int slot = atomicAdd(a.acc.done_count, 1);
                    if (slot < a.acc.done_cap) {
                        a.acc.done_returns[slot] = ep_return;
                        a.acc.done_lengths[slot] = ep_length;
                    }
                    ep_return = 0.0f;
                    ep_length = 0.0f;
                }
            }
            const unsigned long long fin = quad_envs(__ballot(finished));
            wired = ((fin >> e) & 1ull) != 0 ? 1 : wired;
            reset_rows<E>(rows, &was_reset, fin, a.reset_seed + (uint64_t)k * a.reset_stride, env0, lane);
        } else {
            // ---- the draw once more, for the rollout's action and log-probability, which nothing of the step waits for
            const int m = vw - 1;
            detect_sync.arrive();
            if (m == 0 && lane < ne) {
                const int i = env0 + lane;
                const float *lg = logits + lane * (PA_MAX + 1);
                float logp;
                if (GAUSS) {
                    float av[PA_MAX];
                    logp = sample_gaussian(lg, w2a + HEAD_LOG_STD(H), A, sseed, i, av);
                    for (int j = 0; j < A; ++j) a.r_actions[(row + lane) * AW + j] = av[j];
                } else {
                    int sel;
                    sample_categorical_few(lg, A, sseed, i, sel, logp);
                    a.r_actions[row + lane] = (float)sel;
                }
                a.r_logp[row + lane] = logp;
            }
            // ---- critic on the three helpers, at their own barrier
            const int tl = m * WAVE + lane;
            auto critic = [&](auto tiles, int c0) {
                constexpr int NT = decltype(tiles)::value;
                Hidden16Operands<H, IN, NT, KBA> ops;
                ops.load(pc, c0, lane);
                hidden_stack16<H, IN, ACT, NT, KBA, true>(pc, xs, hTc, hTc, ops, c0, lane, critic_sync);
            };
            if (m == 1) critic(std::integral_constant<int, CS.N1>{}, 16 * CS.N0);
            else if (m == 0) critic(std::integral_constant<int, CS.N0>{}, 0);
            else critic(std::integral_constant<int, CS.N2>{}, 16 * (CS.N0 + CS.N1));
            head16_value<H>(w2c, hTc, vals, tl, 3 * WAVE);
        }
        __syncthreads();   // env step done, values complete
        if (tid < ne) a.r_values[row + tid] = vals[tid];
        // a wait that gave up: the block's results are void from here on; leave the loop (every
        // thread reads the same word after the barrier) and end normally
        if (sync_failed != 0u) break;
    }
    if (sync_failed != 0u) {   // nothing of a block whose wait gave up is stored
        if (t == 0) *a.sync_error = 1;
        return;
    }

    if (owner) {
        a.acc.ep_return[env0 + my_env] = ep_return;
        a.acc.ep_length[env0 + my_env] = ep_length;
    }
    for (int i = t; i < nenv * E::OBS; i += T) {
        const int r = i / E::OBS, c = i - r * E::OBS;
        a.obs[(size_t)env0 * E::OBS + i] = rows[r * S::STRIDE + c];
    }
    S::out(rows, gbase, nenv, t, 0, E::STATE);
}

struct CartPoleSlot {
    static constexpr int OBS = cartpole::OBS, ACT_W = 1, HEAD = 2;   // HEAD: outputs of the actor's head
    float s[4];
    int32_t steps;
    MRL_DEV void load(const float *states, const int32_t *side, int i) {
        const float4 v = reinterpret_cast<const float4 *>(states)[i];
        s[0] = v.x; s[1] = v.y; s[2] = v.z; s[3] = v.w;
        steps = side[i];
    }
    MRL_DEV void store(float *states, int32_t *side, int i) const {
        reinterpret_cast<float4 *>(states)[i] = make_float4(s[0], s[1], s[2], s[3]);
        side[i] = steps;
    }
    MRL_DEV float obs(int k) const { return s[k]; }
    MRL_DEV void step(const float *act, float &r, float &d) { cartpole::step(s, steps, (int)act[0], r, d); }
    MRL_DEV void reset(int i, uint64_t seed) { cartpole::reset(s, steps, i, (uint32_t)seed); }
};
struct PendulumSlot {
    static constexpr int OBS = pendulum::OBS, ACT_W = 1, HEAD = 1;
    float s[8];
    MRL_DEV void load(const float *states, const int32_t *, int i) {
        const float4 *row = reinterpret_cast<const float4 *>(states) + 2 * (size_t)i;
        const float4 a = row[0], b = row[1];
        s[0] = a.x; s[1] = a.y; s[2] = a.z; s[3] = a.w; s[4] = b.x; s[5] = b.y; s[6] = b.z; s[7] = b.w;
    }
    MRL_DEV void store(float *states, int32_t *, int i) const {
        float4 *row = reinterpret_cast<float4 *>(states) + 2 * (size_t)i;
        row[0] = make_float4(s[0], s[1], s[2], s[3]);
        row[1] = make_float4(s[4], s[5], s[6], s[7]);
    }
    MRL_DEV float obs(int k) const { return s[k]; }
    MRL_DEV void step(const float *act, float &r, float &d) { pendulum::step(s, act[0], r, d); }
    MRL_DEV void reset(int i, uint64_t seed) { pendulum::reset(s, i, seed); }
};

// ---------------------------------------------------------------- CartPole / Pendulum, 16 rows per workgroup
// A step of these envs is one dependent chain (observation -> two layers on the matrix cores -> head -> sample -> env
// step) of a few thousand cycles, whatever the number of envs.  Sixteen rows per workgroup of eight wavefronts (four
// per net, H / 4 columns each, 16x16x4 tiles: the bits of the 32-row tiles) make its matrix part a quarter of that of
// a 32-row workgroup with two wavefronts per net, the number of head outputs is a compile-time constant, and the
// log-probability, which nothing of the step waits for, is taken by another wavefront beside the env step.  Lanes
// 0 .. 15 of wavefront 0 carry one env each in registers.  Up to hidden width 128 the hidden layers' weights stay in
// registers for the whole launch (the bound of four wavefronts per SIMD lets two workgroups share a CU).
// CartPole, hidden width 64, us per step at 1024 / 4096 envs: 32 rows 4.88 / 4.66, this form 3.04 / 3.11 (2.50 at 1024 envs
// with the head's sums in DPP instructions); hidden width
// 128 and 256 as a policy and an env-step launch per step 16.9 and 19.4, in this form 5.95 and 13.4.  (The critic a
// phase behind the actor, its second layer beside the env step: 3.30 at width 64, 7.2 at 128 -- on one SIMD matrix and
// vector instructions of different wavefronts take turns --, 12.5 at 256.)
template <class C, int H, int ACT, bool GAUSS>
__global__ __launch_bounds__(512, 4) void collect_classic16_kernel(CollectArgs a, int32_t *side) {
    constexpr int IN = C::OBS, AW = C::ACT_W, A = C::HEAD, R = PR16, T = 512, NT = H / 64;
    constexpr bool RESIDENT = H <= 128;
    constexpr int KB = RESIDENT ? H / 4 : 8;   // k-steps of layer-1 weights held (all of them, or the next block)
    __shared__ float xs[R * XS_LD];
    __shared__ float hT[2][H * HT16_LD];
    __shared__ float h2[2][R * (H + 1)];
    __shared__ float logits[R * (PA_MAX + 1)];
    __shared__ float vals[R];
    __shared__ __align__(16) float w2a[HEAD_LDS(H)];
    __shared__ float w2c[H + 1];
    const int t = threadIdx.x;
    const int env0 = blockIdx.x * R;
    const int nenv = min(R, a.n_envs - env0);
    const int N = a.n_envs;
    const bool owner = t < nenv;   // lanes 0 .. nenv - 1 of wavefront 0: one env each
    C slot{};
    float ep_return = 0.0f, ep_length = 0.0f;
    if (owner) {
        slot.load(a.states, side, env0 + t);
        ep_return = a.acc.ep_return[env0 + t];
        ep_length = a.acc.ep_length[env0 + t];
    }
    stage_head(a.actor_p + IN * H + H + H * H + H, H, A, GAUSS, w2a, t, T);
    for (int i = t; i < H + 1; i += T) w2c[i] = a.critic_p[IN * H + H + H * H + H + i];
    for (int i = t; i < R * XS_LD; i += T) xs[i] = 0.0f;
    Hidden16Operands<H, IN, NT, KB> ops;
    if (RESIDENT) ops.load(t >= T / 2 ? a.critic_p : a.actor_p, 16 * NT * ((t / WAVE) & 3), t % WAVE);
    __syncthreads();
    // the policy does not change during the launch: exp(log_std) of the Gaussian head once for all the steps
    float stdv[A];
#pragma unroll
    for (int j = 0; j < A; ++j)
        stdv[j] = GAUSS ? exp32(gaussian_log_std(w2a[HEAD_LOG_STD(H) + j])) : 1.0f;

    for (int k = 0; k < a.n_steps; ++k) {
        // (the empty asm keeps what the optimiser derives from these values inside the step)
        int tid = t, ne = __builtin_amdgcn_readfirstlane(nenv), zero = 0;
        asm volatile("" : "+v"(tid), "+s"(zero), "+s"(ne) : : "memory");
        const int wave = tid / WAVE, lane = tid % WAVE, net = wave >> 2, c0 = 16 * NT * (wave & 3);
        const float *p = (net ? a.critic_p : a.actor_p) + zero;
        const size_t row = (size_t)(a.t0 + k) * N + env0;   // this block's slice of rollout row t
        const uint32_t sseed = a.sample_seed + (uint32_t)k * a.sample_stride;
        if (!RESIDENT) ops.load(p, c0, lane);
        if (tid < ne) {
#pragma unroll
            for (int c = 0; c < IN; ++c) {
                const float v = slot.obs(c);
                xs[tid * XS_LD + c] = v;
                a.r_obs[(row + tid) * IN + c] = v;
            }
        }
        __syncthreads();
        BlockSync bs;
        hidden_stack16<H, IN, ACT, NT, KB, false>(p, xs, hT[net], h2[net], ops, c0, lane, bs);
        if (net == 0) head16<H>(w2a, A, h2[0], logits, PA_MAX + 1, tid, T / 2);
        else head16_value<H>(w2c, h2[1], vals, tid - T / 2, T / 2);
        __syncthreads();
        if (wave > 1 || lane >= ne) continue;
        // wavefronts 0 and 1 draw the action; 1 goes on to its log-probability and the rollout row, 0 to the env step
        const int i = env0 + lane;
        float av[A], logp;
        if (GAUSS) {
            logp = sample_gaussian(logits + lane * (PA_MAX + 1), w2a + HEAD_LOG_STD(H), A, sseed, i, av, stdv);
        } else {
            int sel;
            sample_categorical_few(logits + lane * (PA_MAX + 1), A, sseed, i, sel, logp);
            av[0] = (float)sel;
        }
        if (wave == 1) {
            for (int j = 0; j < AW; ++j) a.r_actions[(row + lane) * AW + j] = av[j];
            a.r_logp[row + lane] = logp;
            a.r_values[row + lane] = vals[lane];
            continue;
        }
        float r, d;
        slot.step(av, r, d);
        a.r_rewards[row + lane] = r;
        a.r_dones[row + lane] = d;
        ep_return = ep_return + r;
        ep_length = ep_length + 1.0f;
        if (d > 0.5f) {
            const int s = atomicAdd(a.acc.done_count, 1);
            if (s < a.acc.done_cap) {
                a.acc.done_returns[s] = ep_return;
                a.acc.done_lengths[s] = ep_length;
            }
            ep_return = 0.0f;
            ep_length = 0.0f;
            slot.reset(i, a.reset_seed + (uint64_t)k * a.reset_stride);
        }
    }
    if (owner) {
        slot.store(a.states, side, env0 + t);
#pragma unroll
        for (int c = 0; c < IN; ++c) a.obs[(size_t)(env0 + t) * IN + c] = slot.obs(c);
        a.acc.ep_return[env0 + t] = ep_return;
        a.acc.ep_length[env0 + t] = ep_length;
    }
}

// the workgroups of `grid` = 16 envs each; side: CartPole's step counters
template <int H, int ACT>
int launch_collect16_t(mrl_ctx *ctx, const mrl_rollout *r, const CollectArgs &a, int32_t *side) {
    const dim3 grid(grid_for(r->n_envs, PR16)), block(LunarLander::THREADS);
    if (r->env_id == MRL_ENV_LUNARLANDER)
        hipLaunchKernelGGL((collect16_kernel<LunarLander, H, ACT, false>), grid, block, 0, ctx->stream, a);
    else if (r->env_id == MRL_ENV_LUNARLANDER_CONTINUOUS)
        hipLaunchKernelGGL((collect16_kernel<LunarLanderContinuous, H, ACT, true>), grid, block, 0, ctx->stream, a);
    else if (r->env_id == MRL_ENV_CARTPOLE)
        hipLaunchKernelGGL((collect_classic16_kernel<CartPoleSlot, H, ACT, false>), grid, dim3(512), 0, ctx->stream, a, side);
    else
        hipLaunchKernelGGL((collect_classic16_kernel<PendulumSlot, H, ACT, true>), grid, dim3(512), 0, ctx->stream, a, side);
    MRL_CHECK_LAUNCH();
    return MRL_OK;
}

}  // namespace mrl
