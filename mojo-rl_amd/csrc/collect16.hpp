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
#include "collect_books.hpp"

namespace mrl {

template <int A, int B>
constexpr int cmax() { return A > B ? A : B; }

// column tiles of 16 of the critic on the three helpers: helper 0, which writes the rollout row, never more than the others
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
//                           env, one per body: env_lunar.hpp), resets;
//   the other three         contact detection, what the engines need whatever the action is, the rollout row of step k - 1 and
//                           the draw's numbers of step k + 1, then the critic (H = 256: 80 / 96 / 80 columns) at a barrier
//                           of their own.
// Two such workgroups fit a CU (LDS, registers).  On this hardware a SIMD issues either a matrix or a vector instruction,
// never both at once (a wavefront of dependent v_fma_f32 that shares its SIMD with a wavefront issuing v_mfma back to back
// takes the sum of both times), so at H = 256 the second one costs what its forward passes cost (4096 : 8192 envs 18.5 :
// 27.3 us per step); still, since the solver carries four lanes per env, two of 16 rows are ahead of one of 32 rows with one
// lane per env and the critic on six wavefronts (33.0).
// One lane per env : four, us per step: 777 envs, H = 64 19.4 : 12.9 (its solver wavefront: 22 of 37 thousand cycles in the
// physics before); 4096 envs, H = 64 18.8 : 12.6, H = 256, where the critic is the longer path, 23.9 : 21.6.  The engines'
// sines and the log-probability off the solver, its detection in one pass of all four wavefronts: H = 64, 777 envs
// 11.46 : 11.26, 4096 envs 11.86 : 11.55 (11.2 since a step's first loads are no longer waited for; thousand cycles of a
// step there: actor 5.0, sample 1.1, detection 3.5, wait 0.8, engines 1.6, physics and tail 12, reset 1).  Numbers of the draw a
// step ahead, rollout rows and episode sums a step later, at 8192 envs, H = 64 / 128 / 256: 14.3 / 16.1 / 27.5 : 14.2 / 15.8 /
// 27.4, two continuous actions 14.8 / 19.2 / 30.5 : 14.4 / 18.7 / 29.8 (means over three to twelve freshly initialised policies; of
// the twelve at 256 ten are faster, by 0.4 to 1.3 %, and two slower, by 1.2: how the two workgroups of a CU fall in with each other).  (32 envs a workgroup of eight wavefronts, a weight operand
// for two row tiles, H = 256: 27.2 at 8192 envs, but 27.0 : 26.1 at 4097 and 53.6 : 44.7 at 9001: matrix and vector time of a
// SIMD add up either way.)
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
    // of step k at [k & 1]: numbers of the draw (there a step ahead), actions, probabilities / means, rewards, done flags, values
    __shared__ float numbers[2][R * AW], acts[2][R * AW], chance[2][R * AW], rew[2][R], don[2][R], vals[2][R];
    __shared__ EpisodeBooks::Waiting listed;
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
    auto make_numbers = [&](int k, int lane) {
        if (lane >= R * AW) return;
        const uint32_t seed = a.sample_seed + (uint32_t)k * a.sample_stride;
        const int i = env0 + lane / AW;
        numbers[k & 1][lane] = GAUSS ? gaussian_noise(seed, i, a.A, lane % AW) : categorical_uniform(seed, i);
    };
    if (t >= T - WAVE) make_numbers(0, t - (T - WAVE));
    __syncthreads();
    // the first helper keeps the episode sums, a lane per env
    const int t_books = t - WAVE * ((sw + 1) & 3);
    EpisodeBooks books;
    books.begin(a, env0 + t_books, t_books >= 0 && t_books < nenv);
    auto book = [&](int k, int lane, int ne) {   // what step k leaves beside the rows
        const size_t at = (size_t)(a.t0 + k) * N + env0 + lane;
        const int q = k & 1, e = lane & (R - 1);
        const bool mine = lane < ne;
        if (mine) {
            float logp = 0.0f;
#pragma unroll
            for (int j = 0; j < AW; ++j) {
                const float u = acts[q][e * AW + j], c = chance[q][e * AW + j];
                a.r_actions[at * AW + j] = u;
                if (GAUSS) {
                    const float log_std = gaussian_log_std(w2a[HEAD_LOG_STD(H) + j]);
                    logp = logp + gaussian_logp(u, c, log_std, exp32(log_std));
                } else {
                    logp = log32(c + 1e-8f);
                }
            }
            a.r_logp[at] = logp;
            a.r_values[at] = vals[q][e];
        }
        books.rewards(a, listed, k, at, rew[q][e], don[q][e], lane, mine);
    };
    // solver wavefront, four lanes per env: what the env's wiring is (E::lanes_wired) in all four
    const int my_env = (t & 63) >> 2;
    const float my_std = GAUSS && (t & 3) < AW ? exp32(gaussian_log_std(w2a[HEAD_LOG_STD(H) + (t & 3)])) : 1.0f;
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
        const int now = k & 1;
        float drawn[2] = {0.0f, 0.0f};
        if (vw == 0) {   // ---- draw
            const int e = lane >> 2, l = lane & 3;
            const float logit = logits[e * (PA_MAX + 1) + (l < A ? l : 0)];
            if (GAUSS) {   // (one component a lane)
                const float u = logit + my_std * numbers[now][e * AW + (l < AW ? l : 0)];
                if (l < AW) {
                    acts[now][e * AW + l] = u;
                    chance[now][e * AW + l] = logit;
                }
                drawn[0] = quad_bcast<0>(u);
                drawn[1] = quad_bcast<1>(u);
            } else {   // (four actions: the entry refuses any other head)
                float pr;
                drawn[0] = (float)sample_categorical_quad(logit, A, numbers[now][e], l, pr);
                if (l == 0) {
                    acts[now][e] = drawn[0];
                    chance[now][e] = pr;
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
            if (first) carry = E::step_begin(rows + e * S::STRIDE, env0 + e, drawn, shapes, draws + e);
            float r = 0.0f, d = 0.0f;
            step_finish_quads<E, CAP>(rows, cts, shapes, dlist, dcount, carry, wired, lane, ne, r, d);
            if (first) {
                rew[now][e] = r;
                don[now][e] = d;
            }
            const bool finished = first && d > 0.5f;
            const unsigned long long fin = quad_envs(__ballot(finished));
            wired = ((fin >> e) & 1ull) != 0 ? 1 : wired;
            reset_rows<E>(rows, &was_reset, fin, a.reset_seed + (uint64_t)k * a.reset_stride, env0, lane);
        } else {
            const int m = vw - 1;
            detect_sync.arrive();
            if (m == 0 && k > 0) book(k - 1, lane, ne);
            if (m == 1) make_numbers(k + 1, lane);
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
            head16_value<H>(w2c, hTc, vals[now], tl, 3 * WAVE);
        }
        __syncthreads();   // env step done, values complete
        // a wait that gave up: the block's results are void from here on; leave the loop (every
        // thread reads the same word after the barrier) and end normally
        if (sync_failed != 0u) break;
    }
    if (sync_failed != 0u) {   // nothing of a block whose wait gave up is stored
        if (t == 0) *a.sync_error = 1;
        return;
    }

    if (t_books >= 0 && t_books < WAVE) {
        if (a.n_steps > 0) book(a.n_steps - 1, t_books, nenv);
        books.end(a, listed, env0 + t_books, t_books, t_books < nenv);
    }
    for (int i = t; i < nenv * E::OBS; i += T) {
        const int r = i / E::OBS, c = i - r * E::OBS;
        a.obs[(size_t)env0 * E::OBS + i] = rows[r * S::STRIDE + c];
    }
    S::out(rows, gbase, nenv, t, 0, E::STATE);
}

// The same with eight wavefronts, for as many envs as leave every CU one workgroup: nothing shares a SIMD with a second
// solver then, and what the solver wavefront's chain does not need in turn has wavefronts of its own.  A step is
//   wavefront 0       actor columns | draw, the lander's push picked | merge, physics, reward | resets
//             1, 2, 3 actor columns | 1: the rollout row of step k - 1; 2: the numbers of the draw of k + 1; 3: engines | ...
//             4 .. 7  contact detection (14 tasks of 16 envs) beside the actor | critic ...
// Up to width 128 wavefront 2, which has none of the critic there, also puts the observations out and makes the rows of all envs
// as if each started again, so that the solver copies one where it used to build it (1.6 thousand cycles a step); at 256 the
// critic is the longer path already (16.0 : 16.2 us per step with the observations on it).
// The engines (double precision) push the lander in one of four ways: wavefront 3 takes all four, a lane per (env, action),
// beside the draw.  (Two continuous actions: its lanes take what the engines need whatever the action is.)  The critic runs
// on wavefronts 5 to 7, at hidden width 256 on 1 to 3 as well: the SIMDs that the solver does not use.  Weights up to width
// 128 stay in registers (wavefront 0, whose solver wants them: width 64).
// us per step, four wavefronts : eight (without those rows): 777 envs, H = 64 11.04 : 8.63 (9.09), H = 128 13.2 : 10.4 (10.8),
// H = 256 18.2 : 15.8; 4096 envs 11.04 : 8.82 (9.09), 13.3 : 10.5 (10.9), 18.5 : 16.0; two continuous actions, 777 envs, 13.0 :
// 10.9, 15.5 : 13.0, 19.9 : 17.0.  Thousand cycles of a step at H = 64 (of 20; 25 with four): actor and draw 3.7, wait for
// detection and engines 1.5, merge, physics and reward 13.1; at H = 256 (35): actor 13.7, draw and wait 3, physics 13, resets
// 1.6, wait for the critic 3.5.
template <class E, int H, int ACT, bool GAUSS>
__global__ __launch_bounds__(512, 2) void collect16_wide_kernel(CollectArgs a) {
    using S = Stage<E>;
    constexpr int IN = E::OBS, AW = E::ACT_W, A = GAUSS ? 2 : 4, R = PR16, T = 512, CAP = 3;
    constexpr int NTA = H / 64, KB = H <= 128 ? H / 4 : 8, KB0 = H == 64 ? KB : 8;   // (wavefront 0's)
    constexpr int K0 = IN / 4, TILES = H / 16;
    constexpr int CW = H == 256 ? 6 : 3;                                             // the critic's wavefronts
    constexpr bool FRESH = H <= 128;   // wavefront 2 has time for new episodes' rows (at 256 it has columns of the critic)
    constexpr unsigned DETECTING = FRESH ? 6 : 5;   // wavefronts 2 (which puts the observations out) .. 7; 3 .. 7
    static_assert(IN % 4 == 0 && E::DETECT_TASKS <= 16, "whole k-steps; detection in one pass of four wavefronts");
    __shared__ float rows[R * S::STRIDE];
    __shared__ float xs[R * XS_LD];
    __shared__ __align__(16) float w2a[HEAD_LDS(H)];
    __shared__ float w2c[H + 1];
    __shared__ float logits[R * (PA_MAX + 1)];
    __shared__ float shapes[E::NSHAPE];
    __shared__ ll::EngineDraw draws[R];
    __shared__ ll::Velocity pushes[R][4];
    __shared__ unsigned long long was_reset;
    __shared__ unsigned sync_actor, sync_critic, sync_detect, sync_fresh, sync_failed, give_up[2];
    __shared__ float hT[2][H * HT16_LD], h2[2][R * (H + 1)];
    __shared__ float cts[R * S::CSTRIDE], dlist[detect_list_floats<E, CAP>() + 1];
    __shared__ int dcount[detect_count_ints<E>()];
    // of step k at [k & 1]: numbers of the draw (there a step ahead), actions, probabilities / means, rewards, done flags, values
    __shared__ float numbers[2][R * AW], acts[2][R * AW], chance[2][R * AW], rew[2][R], don[2][R], vals[2][R];
    __shared__ EpisodeBooks::Waiting finished;
    __shared__ float fresh[FRESH ? R * S::STRIDE : 1];   // the rows of envs that start again behind this step

    const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t / WAVE);
    const int env0 = blockIdx.x * R;
    const int nenv = min(R, a.n_envs - env0);
    const int N = a.n_envs;
    float *gbase = a.states + (size_t)env0 * E::STATE;
    const size_t row0 = (size_t)a.t0 * N + env0;   // the first step's rollout row

    if (t < E::THREADS) S::in(rows, gbase, nenv, t);
    for (int i = t; i < E::NSHAPE; i += T) shapes[i] = a.shapes[i];
    stage_head(a.actor_p + IN * H + H + H * H + H, H, A, GAUSS, w2a, t, T);
    for (int i = t; i < H + 1; i += T) w2c[i] = a.critic_p[IN * H + H + H * H + H + i];
    auto make_numbers = [&](int k, int lane) {
        if (lane >= R * AW) return;
        const uint32_t seed = a.sample_seed + (uint32_t)k * a.sample_stride;
        const int i = env0 + lane / AW;
        numbers[k & 1][lane] = GAUSS ? gaussian_noise(seed, i, A, lane % AW) : categorical_uniform(seed, i);
    };
    if (wave == 2) make_numbers(0, t % WAVE);
    if (t == 0) {
        was_reset = 0;
        sync_actor = sync_critic = sync_detect = sync_fresh = sync_failed = 0;
        give_up[0] = give_up[1] = 0;
    }
    __syncthreads();

    // Every role counts the same steps, and all meet at the barrier that ends one.  The wavefront-group barriers' counts follow
    // from the step's number.
    constexpr unsigned ACTOR_MEETS = H == 256 ? 3 : 2;
    auto actor_sync = [&](int k) { return WaveGroupSync{&sync_actor, (unsigned)k * 4u * ACTOR_MEETS, 4u, &sync_failed, a.spin_limit}; };
    auto critic_sync = [&](int k) { return WaveGroupSync{&sync_critic, (unsigned)k * 2u * CW, (unsigned)CW, &sync_failed, a.spin_limit}; };
    auto detect_sync = [&](int k) { return WaveGroupSync{&sync_detect, (unsigned)k * DETECTING, DETECTING, &sync_failed, a.spin_limit}; };
    auto fresh_sync = [&](int k) { return WaveGroupSync{&sync_fresh, (unsigned)k, 1u, &sync_failed, a.spin_limit}; };
    // actor: layers on wavefronts 0 .. 3; at width 256 the head as well, into `logits`
    auto actor = [&](auto &ops, const float *pa, int k, int tid) {
        const int lane = tid % WAVE, n = lane & 15, g = lane >> 4, c0 = 16 * NTA * (tid / WAVE);
        float a0[K0];
#pragma unroll
        for (int kk = 0; kk < K0; ++kk) a0[kk] = rows[n * S::STRIDE + 4 * kk + g];
        WaveGroupSync sync = actor_sync(k);
        hidden16_layer0_of<H, IN, ACT>(a0, hT[0], ops, c0, lane);
        sync();
        hidden16_layer1<H, IN, ACT>(pa, hT[0], h2[0], ops, c0, lane, [] {});
        sync();
        if constexpr (H == 256) {
            head16<H>(w2a, A, h2[0], logits, PA_MAX + 1, tid, 4 * WAVE);
            sync();
        }
    };
    // critic, on the wavefronts m = 0 .. CW - 1 of its own: once the observations are out, which detection's barrier tells
    auto critic = [&](auto &ops, const float *pc, int k, int m, int c0, int lane) {
        WaveGroupSync detect = detect_sync(k), sync = critic_sync(k);
        detect.wait_for(detect.target + detect.nwaves);
        hidden16_layer0<H, IN, ACT>(xs, hT[1], ops, c0, lane);
        sync();
        hidden16_layer1<H, IN, ACT>(pc, hT[1], h2[1], ops, c0, lane, [] {});
        sync();
        head16_value<H>(w2c, h2[1], vals[k & 1], m * WAVE + lane, CW * WAVE);
    };
    // A wait that gave up voids the workgroup's results: all leave behind the same barrier, which wavefront 0 decides ahead of it.
    auto step_end = [&](int k) {
        __syncthreads();
        return give_up[k & 1] != 0u;
    };

    if (wave == 0) {
        const int lane0 = t;
        int wired = lane0 >> 2 < nenv ? E::lanes_wired(rows + (lane0 >> 2) * S::STRIDE) : 0;
        Hidden16Operands<H, IN, NTA, KB0> ops;
        if (H == 64) ops.load(a.actor_p, 0, lane0);
        const float std = GAUSS && (lane0 & 3) < A ? exp32(gaussian_log_std(w2a[HEAD_LOG_STD(H) + (lane0 & 3)])) : 1.0f;
        for (int k = 0; k < a.n_steps; ++k) {
            // (Nothing but the rows is carried from one step to the next: the empty asm keeps what the optimiser derives from
            // these values out of the registers that the solver needs.)
            int lane = lane0, ne = __builtin_amdgcn_readfirstlane(nenv), zero = 0;
            asm volatile("" : "+v"(lane), "+s"(zero), "+s"(ne) : : "memory");
            const float *pa = a.actor_p + zero;
            const int e = lane >> 2, l = lane & 3, now = k & 1;
            float *row = rows + e * S::STRIDE;
            if (H != 64) ops.load(pa, 0, lane);
            actor(ops, pa, k, lane);
            float mine;
            if constexpr (H == 64) {
                float out[4];
                head_row16<H, 4, PA_MAX>(w2a, h2[0], e, l, out);
                mine = l == 0 ? out[0] : l == 1 ? out[1] : l == 2 ? out[2] : out[3];
            } else {
                if (H == 128) {
                    head16<H>(w2a, A, h2[0], logits, PA_MAX + 1, lane, WAVE);
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");   // (this wavefront's own writes)
                }
                mine = logits[e * (PA_MAX + 1) + (l < A ? l : 0)];
            }
            WaveGroupSync detect = detect_sync(k);
            typename E::Carry carry{};
            const bool first = l == 0 && e < ne;
            if constexpr (GAUSS) {
                const float u = mine + std * numbers[now][e * AW + (l < A ? l : 0)];
                if (l < A) {
                    acts[now][e * AW + l] = u;
                    chance[now][e * AW + l] = mine;
                }
                const float both[2] = {quad_bcast<0>(u), quad_bcast<1>(u)};
                detect.wait_for(detect.target + detect.nwaves);
                if (first) carry = E::step_begin(row, env0 + e, both, shapes, draws + e);
            } else {
                float pr;
                const int sel = sample_categorical_quad(mine, A, numbers[now][e], l, pr);
                if (l == 0) {
                    acts[now][e] = (float)sel;
                    chance[now][e] = pr;
                }
                detect.wait_for(detect.target + detect.nwaves);
                if (first) carry = ll::step_begin_pushed(row, sel, pushes[e][sel]);
            }
            float r = 0.0f, d = 0.0f;
            step_finish_quads<E, CAP>(rows, cts, shapes, dlist, dcount, carry, wired, lane, ne, r, d);
            const bool over = first && d > 0.5f;
            if (first) {
                rew[now][e] = r;
                don[now][e] = d;
            }
            const unsigned long long fin = quad_envs(__ballot(over));
            wired = ((fin >> e) & 1ull) != 0 ? 1 : wired;
            if constexpr (FRESH) {
                if (fin != 0) {
                    WaveGroupSync made = fresh_sync(k);
                    made.wait_for(made.target + made.nwaves);
                }
                for (unsigned long long m = fin; m; m &= m - 1) {
                    const int at = (__ffsll((long long)m) - 1) * S::STRIDE;
#pragma unroll
                    for (int c = lane; c < E::STATE; c += WAVE) rows[at + c] = fresh[at + c];
                }
            } else {
                reset_rows<E>(rows, &was_reset, fin, a.reset_seed + (uint64_t)k * a.reset_stride, env0, lane);
            }
            if (lane == 0) give_up[now] = __hip_atomic_load(&sync_failed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            if (step_end(k)) break;
        }
    } else if (wave < 4) {
        const int lane0 = t % WAVE;
        Hidden16Operands<H, IN, NTA, KB> ops;
        if (H <= 128) ops.load(a.actor_p, 16 * NTA * wave, lane0);
        EpisodeBooks books;
        const bool mine = wave == 1 && lane0 < nenv;
        books.begin(a, env0 + lane0, mine);
        float log_std[AW], std[AW];
#pragma unroll
        for (int j = 0; j < AW; ++j) {
            log_std[j] = GAUSS ? gaussian_log_std(w2a[HEAD_LOG_STD(H) + j]) : 0.0f;
            std[j] = GAUSS ? exp32(log_std[j]) : 1.0f;
        }
        auto book = [&](int k, int lane) {   // what step k leaves beside the rows
            const size_t at = row0 + (size_t)k * N + lane;
            const int q = k & 1, e = lane & (R - 1);
            if (mine) {
                float logp = 0.0f;
#pragma unroll
                for (int j = 0; j < AW; ++j) {
                    const float u = acts[q][e * AW + j], c = chance[q][e * AW + j];
                    a.r_actions[at * AW + j] = u;
                    if (GAUSS) logp = logp + gaussian_logp(u, c, log_std[j], std[j]);
                    else logp = log32(c + 1e-8f);
                }
                a.r_logp[at] = logp;
                a.r_values[at] = vals[q][e];
            }
            books.rewards(a, finished, k, at, rew[q][e], don[q][e], lane, mine);
        };
        int done = 0;   // steps taken
        for (int k = 0; k < a.n_steps; ++k) {
            int lane = lane0, ne = __builtin_amdgcn_readfirstlane(nenv), zero = 0;
            asm volatile("" : "+v"(lane), "+s"(zero), "+s"(ne) : : "memory");
            const float *pa = a.actor_p + zero, *pc = a.critic_p + zero;
            if (H == 256) ops.load(pa, 16 * NTA * wave, lane);
            actor(ops, pa, k, wave * WAVE + lane);
            if (wave == 1) {
                if (k > 0) book(k - 1, lane);
            } else if (wave == 2) {
                if constexpr (FRESH) {
                    stage_observations<IN, WAVE>(xs, a.r_obs + (row0 + (size_t)k * N) * IN, ne, lane,
                                                 [&](int r, int c) { return rows[r * S::STRIDE + c]; });
                    detect_sync(k).arrive();
                }
                make_numbers(k + 1, lane);
                if constexpr (FRESH) {
                    const int e = lane >> 2;
                    const uint64_t seed = a.reset_seed + (uint64_t)k * a.reset_stride;
                    ll::reset_row_quad(fresh + e * S::STRIDE, ll::combined_seed(seed, env0 + e), lane & 3);
                    fresh_sync(k).arrive();
                }
            } else {
                const int e = GAUSS ? lane : lane >> 2;
                if (e < nenv) {
                    const float *row = rows + e * S::STRIDE;
                    if constexpr (GAUSS) draws[e] = ll::engine_draw(row, env0 + e);
                    else pushes[e][lane & 3] = ll::pushed(row, env0 + e, lane & 3, shapes);
                }
                detect_sync(k).arrive();
            }
            if constexpr (H == 256) {   // (columns: 1, 2, 1 of the sixteen tiles here, four on each of the others)
                auto share = [&](auto tiles, int m, int c0) {
                    Hidden16Operands<H, IN, decltype(tiles)::value, 8> cops;
                    cops.load(pc, c0, lane);
                    critic(cops, pc, k, m, c0, lane);
                };
                if (wave == 2) share(std::integral_constant<int, 2>{}, 1, 16);
                else share(std::integral_constant<int, 1>{}, wave - 1, wave == 1 ? 0 : 48);
            }
            done = k + 1;
            if (step_end(k)) break;
        }
        if (wave == 1 && sync_failed == 0u) {
            if (done > 0) book(done - 1, lane0);
            books.end(a, finished, env0 + lane0, lane0, mine);
        }
    } else {
        const int lane0 = t % WAVE, v = wave - 4;
        auto helper = [&](auto tiles, int m, int c0) {
            constexpr int NT = decltype(tiles)::value;
            Hidden16Operands<H, IN, NT == 0 ? 1 : NT, KB> ops;
            if (NT > 0 && H <= 128) ops.load(a.critic_p, c0, lane0);
            for (int k = 0; k < a.n_steps; ++k) {
                int lane = lane0, ne = __builtin_amdgcn_readfirstlane(nenv), zero = 0;
                asm volatile("" : "+v"(lane), "+s"(zero), "+s"(ne) : : "memory");
                const float *pc = a.critic_p + zero;
                if constexpr (!FRESH)
                    stage_observations<IN, 4 * WAVE>(xs, a.r_obs + (row0 + (size_t)k * N) * IN, ne, v * WAVE + lane,
                                                     [&](int r, int c) { return rows[r * S::STRIDE + c]; });
                const int task = 4 * v + lane / R, e = lane % R;
                if (task < E::DETECT_TASKS && e < ne) detect_vertex_task<E, CAP>(rows, shapes, dlist, dcount, task, e);
                detect_sync(k).arrive();
                if constexpr (NT > 0) {
                    if (H == 256) ops.load(pc, c0, lane);
                    critic(ops, pc, k, m, c0, lane);
                }
                if (step_end(k)) break;
            }
        };
        // (wavefront 4 has the solver's SIMD)
        constexpr int C0 = H == 256 ? 4 : 0, N0 = (TILES - C0) / 3, N1 = (TILES - C0 - N0) / 2, N2 = TILES - C0 - N0 - N1;
        static_assert(C0 + N0 + N1 + N2 == TILES, "all of the critic's columns");
        if (v == 0) helper(std::integral_constant<int, 0>{}, 0, 0);
        else if (v == 1) helper(std::integral_constant<int, N0>{}, CW - 3, 16 * C0);
        else if (v == 2) helper(std::integral_constant<int, N1>{}, CW - 2, 16 * (C0 + N0));
        else helper(std::integral_constant<int, N2>{}, CW - 1, 16 * (C0 + N0 + N1));
    }
    __syncthreads();
    if (sync_failed != 0u) {   // nothing of a workgroup whose wait gave up is stored
        if (t == 0) *a.sync_error = 1;
        return;
    }
    for (int i = t; i < nenv * E::OBS; i += T) {
        const int r = i / E::OBS, c = i - r * E::OBS;
        a.obs[(size_t)env0 * E::OBS + i] = rows[r * S::STRIDE + c];
    }
    if (t < E::THREADS) S::out(rows, gbase, nenv, t, 0, E::STATE);
}

struct PendulumSlot {
    static constexpr int OBS = pendulum::OBS;
    float s[8];
    MRL_DEV void load(const float *states, int i) {
        const float4 *row = reinterpret_cast<const float4 *>(states) + 2 * (size_t)i;
        const float4 a = row[0], b = row[1];
        s[0] = a.x; s[1] = a.y; s[2] = a.z; s[3] = a.w; s[4] = b.x; s[5] = b.y; s[6] = b.z; s[7] = b.w;
    }
    MRL_DEV void store(float *states, int i) const {
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
// a 32-row workgroup with two wavefronts per net, and the number of head outputs is a compile-time constant.  Up to
// hidden width 128 the hidden layers' weights stay in registers for the whole launch (the bound of four wavefronts per
// SIMD lets two workgroups share a CU).  What a step does not need in turn is not in the chain:
//   * CartPole has two actions: while wavefront 0 takes the actor's head and draws, wavefront 5 takes the env step with
//     both, and the draw picks one of two rows;
//   * the states of envs that start again (wavefront 6), the uniform numbers of the draw (2) and Pendulum's normal
//     numbers (2) depend on seeds alone: each is there a step ahead;
//   * log-probability, rollout row and episode sums are taken a step later (CartPole), or beside the env step (Pendulum).
// (The critic a phase behind the actor where it has the actor's SIMDs: slower at widths 64 and 128 -- on one SIMD matrix and
// vector instructions of different wavefronts take turns; width 64 gives it two SIMDs that the draw does not use.)
// A step's chain waits for its longest wavefront at three barriers; thousand cycles of CartPole's at width 64 and 1024 envs,
// with all of it in turn 5.9 in four barriers, now 3.1: layer 0 0.6, layer 1 1.2, head and draw (beside the critic's
// second layer) 1.3.  us per step before : now, CartPole at 1024 / 4096 / 8192 / 16384 / 32768 envs 2.55 : 1.36, 2.65 : 1.42,
// 4.25 : 2.12, 5.91 : 4.10, 14.3 : 8.0; width 128, 1024 envs 5.66 : 4.59; width 256 10.5 : 10.4.  Pendulum at 1024 / 8192 /
// 16384 / 32768 envs 2.77 : 1.86, 3.92 : 3.08, 6.22 : 5.87, 12.0 : 11.4; width 128, 1024 envs 6.36 : 6.07; width 256 11.8 :
// 11.3.  (From 8192 CartPole and 16384 Pendulum envs on, before, in 32-row workgroups with one env a lane in turn.)
// What a CartPole workgroup has in LDS beside its nets.  The envs' rows behind the last step, one per action and env: a new
// episode's where that action ended one.  Of step k, at [k & 1]: the action drawn, its probability, both actions' rewards and
// done flags; and, there a step ahead, new episodes' rows and the numbers of the draw.
struct CartPoleRows {
    static constexpr int R = PR16, A = 2, SLD = 5;
    float rows[A][R][SLD];
    int32_t steps[A][R];
    float rew[2][A][R], don[2][A][R], prob[2][R];
    int32_t drawn[2][R];
    float fresh[2][R][SLD], uniform[2][R];

    // as if a step with action 0 had led here; lanes 0 .. R - 1
    MRL_DEV void load(const CollectArgs &a, const int32_t *side, int env0, int nenv, int e) {
        float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        int32_t n = 0;
        if (e < nenv) {
            v = reinterpret_cast<const float4 *>(a.states)[env0 + e];
            n = side[env0 + e];
        }
#pragma unroll
        for (int j = 0; j < A; ++j) {
            rows[j][e][0] = v.x; rows[j][e][1] = v.y; rows[j][e][2] = v.z; rows[j][e][3] = v.w;
            steps[j][e] = n;
        }
        drawn[1][e] = 0;
    }
    MRL_DEV void store(const CollectArgs &a, int32_t *side, int env0, int e) const {
        const int sel = drawn[(a.n_steps + 1) & 1][e];
        const float *s = rows[sel][e];
        reinterpret_cast<float4 *>(a.states)[env0 + e] = make_float4(s[0], s[1], s[2], s[3]);
        side[env0 + e] = steps[sel][e];
#pragma unroll
        for (int c = 0; c < 4; ++c) a.obs[(size_t)(env0 + e) * 4 + c] = s[c];
    }
    // the operand of layer 0: input `lane >> 4` of row `lane & 15`
    MRL_DEV float input(int before, int lane) const {
        const int n = lane & 15, g = lane >> 4, sel = drawn[before][n];
        const float x0 = rows[0][n][g], x1 = rows[1][n][g];
        return sel != 0 ? x1 : x0;
    }
    MRL_DEV void make_fresh(const CollectArgs &a, int k, int env0, int e) {
        float s[4];
        int32_t none;
        cartpole::reset(s, none, env0 + e, (uint32_t)(a.reset_seed + (uint64_t)k * a.reset_stride));
#pragma unroll
        for (int c = 0; c < 4; ++c) fresh[k & 1][e][c] = s[c];
    }
    MRL_DEV void make_uniform(const CollectArgs &a, int k, int env0, int e) {
        uniform[k & 1][e] = categorical_uniform(a.sample_seed + (uint32_t)k * a.sample_stride, env0 + e);
    }
    MRL_DEV void book(EpisodeBooks &b, const CollectArgs &a, EpisodeBooks::Waiting &w, int k, size_t at, int lane, bool mine) const {
        const int q = k & 1, e = lane & (R - 1), sel = drawn[q][e];
        if (mine) a.r_actions[at] = (float)sel;
        b.rewards(a, w, k, at, rew[q][sel][e], don[q][sel][e], lane, mine);
    }
    MRL_DEV void draw(int now, int e, int l, float logit) {
        float pr;
        const int sel = sample_categorical_quad(logit, A, uniform[now][e], l, pr);
        if (l == 0) {
            drawn[now][e] = sel;
            prob[now][e] = pr;
        }
    }
};

// The env step of one wavefront, lanes 0 .. 15 with action 0, 16 .. 31 with action 1 (the others repeat them), in three
// pieces that a caller may place at either side of a barrier.
struct CartPoleStep {
    float s[4], again[4];
    cartpole::Push push;
    int32_t n;
    MRL_DEV void begin(const CartPoleRows &c, const CollectArgs &a, size_t row, int ne, int now, int lane) {
        const int e = lane & 15, from = c.drawn[now ^ 1][e];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            s[j] = c.rows[from][e][j];
            again[j] = c.fresh[now][e][j];
        }
        n = c.steps[from][e];
        if (lane < ne) {
#pragma unroll
            for (int j = 0; j < 4; ++j) a.r_obs[(row + lane) * 4 + j] = s[j];
        }
    }
    MRL_DEV void middle(int lane) {
        push = cartpole::push(s, (lane >> 4) & 1);
        asm volatile("" : "+v"(push.sintheta), "+v"(push.costheta), "+v"(push.temp));   // (here, not where they are used)
    }
    MRL_DEV void end(CartPoleRows &c, int now, int lane) {
        const int e = lane & 15, act = (lane >> 4) & 1;
        float r, d;
        cartpole::step(s, n, push, r, d);
        if (lane < 32) {
#pragma unroll
            for (int j = 0; j < 4; ++j) c.rows[act][e][j] = d > 0.5f ? again[j] : s[j];
            c.steps[act][e] = d > 0.5f ? 0 : n;
            c.rew[now][act][e] = r;
            c.don[now][act][e] = d;
        }
    }
};

// Hidden widths 128 and 256: four wavefronts per net.
template <int H, int ACT>
__global__ __launch_bounds__(512, 4) void collect_cartpole16_kernel(CollectArgs a, int32_t *side) {
    constexpr int IN = cartpole::OBS, A = 2, R = PR16, T = 512, NT = H / 64;
    constexpr bool RESIDENT = H <= 128;
    constexpr int KB = RESIDENT ? H / 4 : 8;   // k-steps of layer-1 weights held (all of them, or the next block)
    __shared__ CartPoleRows c;
    __shared__ float vals[2][R];
    __shared__ float hT[2][H * HT16_LD];
    __shared__ float h2[2][R * (H + 1)];
    __shared__ float logits[R * (PA_MAX + 1)];
    __shared__ __align__(16) float w2a[HEAD_LDS(H)];
    __shared__ float w2c[H + 1];
    const int t = threadIdx.x;
    const int env0 = blockIdx.x * R;
    const int nenv = min(R, a.n_envs - env0);
    const int N = a.n_envs;
    __shared__ EpisodeBooks::Waiting finished;
    const bool keeper = t / WAVE == 1;   // wavefront 1, a lane per env
    EpisodeBooks books;
    books.begin(a, env0 + t - WAVE, keeper && t - WAVE < nenv);
    if (t < R) {
        c.load(a, side, env0, nenv, t);
        c.make_fresh(a, 0, env0, t);
        c.make_uniform(a, 0, env0, t);
    }
    stage_head(a.actor_p + IN * H + H + H * H + H, H, A, false, w2a, t, T);
    for (int i = t; i < H + 1; i += T) w2c[i] = a.critic_p[IN * H + H + H * H + H + i];
    Hidden16Operands<H, IN, NT, KB> ops;
    if (RESIDENT) ops.load(t >= T / 2 ? a.critic_p : a.actor_p, 16 * NT * ((t / WAVE) & 3), t % WAVE);
    __syncthreads();

    auto book = [&](int k, int e, int ne) {   // what step k leaves beside the envs' rows
        const size_t at = (size_t)(a.t0 + k) * N + env0 + e;
        c.book(books, a, finished, k, at, e, e < ne);
        if (e >= ne) return;
        a.r_logp[at] = log32(c.prob[k & 1][e] + 1e-8f);
        a.r_values[at] = vals[k & 1][e];
    };
    for (int k = 0; k < a.n_steps; ++k) {
        // (the empty asm keeps what the optimiser derives from these values inside the step)
        int tid = t, ne = __builtin_amdgcn_readfirstlane(nenv), zero = 0;
        asm volatile("" : "+v"(tid), "+s"(zero), "+s"(ne) : : "memory");
        const int wave = tid / WAVE, lane = tid % WAVE, net = wave >> 2, c0 = 16 * NT * (wave & 3);
        const int now = k & 1, before = now ^ 1;
        const float *p = (net ? a.critic_p : a.actor_p) + zero;
        if (!RESIDENT) ops.load(p, c0, lane);
        const float a0[1] = {c.input(before, lane)};
        hidden16_layer0_of<H, IN, ACT, NT, KB>(a0, hT[net], ops, c0, lane);
        __syncthreads();
        hidden16_layer1<H, IN, ACT, NT, KB>(p, hT[net], h2[net], ops, c0, lane, [] {});
        __syncthreads();
        // ---- heads (hidden width 256: on all wavefronts of the net; 128: the actor's on 0, the critic's on 7) and draw
        if (H == 256) {
            if (net == 0) head16<H>(w2a, A, h2[0], logits, PA_MAX + 1, tid, T / 2);
            else head16_value<H>(w2c, h2[1], vals[now], tid - T / 2, T / 2);
            __syncthreads();
        } else if (wave == 7) {
            head16_value<H>(w2c, h2[1], vals[now], lane, WAVE);
        }
        if (wave == 0) {
            const int e = lane >> 2, l = lane & 3;
            if (H != 256) {
                head16<H>(w2a, A, h2[0], logits, PA_MAX + 1, lane, WAVE);
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");   // (this wavefront's own writes)
            }
            c.draw(now, e, l, logits[e * (PA_MAX + 1) + (l & 1)]);
        } else if (wave == 5) {
            CartPoleStep step;
            step.begin(c, a, (size_t)(a.t0 + k) * N + env0, ne, now, lane);
            step.middle(lane);
            step.end(c, now, lane);
        } else if (wave == 1) {
            if (k > 0) book(k - 1, lane, ne);
        } else if (wave == 2) {
            if (lane < R) c.make_uniform(a, k + 1, env0, lane);
        } else if (wave == 3) {
            if (lane < R) c.make_fresh(a, k + 1, env0, lane);
        }
        __syncthreads();
    }
    if (keeper) {
        if (a.n_steps > 0) book(a.n_steps - 1, t - WAVE, nenv);
        books.end(a, finished, env0 + t - WAVE, t - WAVE, t - WAVE < nenv);
    }
    if (t < nenv) c.store(a, side, env0, t);
}

// Hidden width 64.  The critic's products are as long as the actor's and nothing of a step waits for the value, so the
// critic has two wavefronts of its own, on SIMDs 2 and 3, which take its second layer while wavefront 0 draws; its head follows a
// step later.  The chain of a step is the actor's: layer 0 | layer 1 | head and draw.
//   wavefronts 0 .. 3   layer 0           layer 1              0: head, draw; 1: what step k + 1 needs of its seeds
//              4        rewards of k - 1  critic's head k - 1  log-probability of k - 1
//              5        rows              the env step ...     ... with both actions
//              6, 7     critic's layer 0  critic's layer 1 ... ...
template <int ACT>
__global__ __launch_bounds__(512, 4) void collect_cartpole16_h64_kernel(CollectArgs a, int32_t *side) {
    constexpr int H = 64, IN = cartpole::OBS, A = 2, R = PR16, T = 512, KB = H / 4;
    constexpr int EARLY = 8;   // k-steps of the critic's layer 1 beside the actor's (2, 4, 7: 1.35, 1.33, 1.31 us per step)
    __shared__ CartPoleRows c;
    __shared__ float hT[2][H * HT16_LD];
    __shared__ float h2[2][R * (H + 1)];
    __shared__ __align__(16) float w2a[HEAD_LDS(H)];
    __shared__ float w2c[H + 1];
    __shared__ EpisodeBooks::Waiting finished;
    const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t / WAVE), lane = t % WAVE;
    const int env0 = blockIdx.x * R;
    const int nenv = min(R, a.n_envs - env0);
    const int N = a.n_envs;
    if (t < R) {
        c.load(a, side, env0, nenv, t);
        c.make_fresh(a, 0, env0, t);
        c.make_uniform(a, 0, env0, t);
    }
    stage_head(a.actor_p + IN * H + H + H * H + H, H, A, false, w2a, t, T);
    for (int i = t; i < H + 1; i += T) w2c[i] = a.critic_p[IN * H + H + H * H + H + i];
    const bool last = a.n_steps > 0;
    const size_t row0 = (size_t)a.t0 * N + env0;   // the first step's rollout row
    if (wave < 4) {
        Hidden16Operands<H, IN, 1, KB> ops;
        const int c0 = 16 * wave;
        ops.load(a.actor_p, c0, lane);
        __syncthreads();
        const int e = lane >> 2, l = lane & 3;
        HeadRow16<H, A, PA_MAX> head;
        head.load(w2a, l);
        for (int k = 0; k < a.n_steps; ++k) {
            const int now = k & 1;
            const float a0[1] = {c.input(now ^ 1, lane)};
            hidden16_layer0_of<H, IN, ACT, 1, KB>(a0, hT[0], ops, c0, lane);
            __syncthreads();
            floatx4 p[1] = {floatx4{0}};
            hidden16_layer1_steps<H, 0, KB>(hT[0], ops, p, lane);
            hidden16_layer1_end<H, IN, ACT, 1, KB>(p, h2[0], ops, c0, lane);
            __syncthreads();
            if (wave == 0) {
                float out[A];
                head.sums(h2[0], e, l, out);   // (in all four lanes of a row)
                c.draw(now, e, l, l == 0 ? out[0] : out[1]);
            } else if (wave == 1 && lane < R) {
                c.make_uniform(a, k + 1, env0, lane);
                c.make_fresh(a, k + 1, env0, lane);
            }
            __syncthreads();
        }
    } else if (wave == 4) {
        const bool mine = lane < nenv;
        EpisodeBooks books;
        books.begin(a, env0 + lane, mine);
        __syncthreads();
        HeadRow16<H, 1, 1> head;
        head.load(w2c, lane & 3);
        float prob = 0.0f;
        auto rewards = [&](int k) {
            c.book(books, a, finished, k, row0 + (size_t)k * N + lane, lane, mine);
            prob = c.prob[k & 1][lane & (R - 1)];
        };
        auto value = [&](int k) {
            float out[1];
            head.sums(h2[1], lane >> 2, lane & 3, out);
            if ((lane & 3) == 0 && lane >> 2 < nenv) a.r_values[row0 + (size_t)k * N + (lane >> 2)] = out[0];
        };
        auto logp = [&](int k) {
            if (mine) a.r_logp[row0 + (size_t)k * N + lane] = log32(prob + 1e-8f);
        };
        for (int k = 0; k < a.n_steps; ++k) {
            if (k > 0) rewards(k - 1);
            __syncthreads();
            if (k > 0) value(k - 1);
            __syncthreads();
            if (k > 0) logp(k - 1);
            __syncthreads();
        }
        if (last) {
            rewards(a.n_steps - 1);
            value(a.n_steps - 1);
            logp(a.n_steps - 1);
        }
        books.end(a, finished, env0 + lane, lane, mine);
    } else if (wave == 5) {
        __syncthreads();
        for (int k = 0; k < a.n_steps; ++k) {
            CartPoleStep step;
            step.begin(c, a, row0 + (size_t)k * N, nenv, k & 1, lane);
            __syncthreads();
            step.middle(lane);
            __syncthreads();
            step.end(c, k & 1, lane);
            __syncthreads();
        }
        if (lane < nenv) c.store(a, side, env0, lane);
    } else {
        Hidden16Operands<H, IN, 2, KB> ops;
        const int c0 = 32 * (wave - 6);
        ops.load(a.critic_p, c0, lane);
        __syncthreads();
        for (int k = 0; k < a.n_steps; ++k) {
            const float a0[1] = {c.input((k & 1) ^ 1, lane)};
            hidden16_layer0_of<H, IN, ACT, 2, KB>(a0, hT[1], ops, c0, lane);
            __syncthreads();
            floatx4 p[2] = {floatx4{0}, floatx4{0}};
            hidden16_layer1_steps<H, 0, EARLY>(hT[1], ops, p, lane);
            __syncthreads();
            hidden16_layer1_steps<H, EARLY, KB>(hT[1], ops, p, lane);
            hidden16_layer1_end<H, IN, ACT, 2, KB>(p, h2[1], ops, c0, lane);
            __syncthreads();
        }
    }
}

// Lanes 0 .. 15 of wavefront 0 carry one env each in registers.
template <int H, int ACT>
__global__ __launch_bounds__(512, 4) void collect_pendulum16_kernel(CollectArgs a) {
    constexpr int IN = PendulumSlot::OBS, A = 1, R = PR16, T = 512, NT = H / 64;
    constexpr bool RESIDENT = H <= 128;
    constexpr int KB = RESIDENT ? H / 4 : 8;   // k-steps of layer-1 weights held (all of them, or the next block)
    __shared__ float xs[R * XS_LD];
    __shared__ float hT[2][H * HT16_LD];
    __shared__ float h2[2][R * (H + 1)];
    __shared__ float logits[R * (PA_MAX + 1)];
    __shared__ float vals[R];
    __shared__ float noise[2][R];     // step k's normal numbers at [k & 1]
    __shared__ __align__(16) float w2a[HEAD_LDS(H)];
    __shared__ float w2c[H + 1];
    const int t = threadIdx.x;
    const int env0 = blockIdx.x * R;
    const int nenv = min(R, a.n_envs - env0);
    const int N = a.n_envs;
    const bool owner = t < nenv;   // lanes 0 .. nenv - 1 of wavefront 0: one env each
    PendulumSlot slot{};
    float ep_return = 0.0f, ep_length = 0.0f;
    if (owner) {
        slot.load(a.states, env0 + t);
        ep_return = a.acc.ep_return[env0 + t];
        ep_length = a.acc.ep_length[env0 + t];
    }
    stage_head(a.actor_p + IN * H + H + H * H + H, H, A, true, w2a, t, T);
    for (int i = t; i < H + 1; i += T) w2c[i] = a.critic_p[IN * H + H + H * H + H + i];
    for (int i = t; i < R * XS_LD; i += T) xs[i] = 0.0f;
    Hidden16Operands<H, IN, NT, KB> ops;
    if (RESIDENT) ops.load(t >= T / 2 ? a.critic_p : a.actor_p, 16 * NT * ((t / WAVE) & 3), t % WAVE);
    if (t / WAVE == 2 && t % WAVE < R) noise[0][t % WAVE] = gaussian_noise(a.sample_seed, env0 + t % WAVE, A, 0);
    __syncthreads();
    // the policy does not change during the launch: exp(log_std) of the Gaussian head once for all the steps
    const float stdv = exp32(gaussian_log_std(w2a[HEAD_LOG_STD(H)]));

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
        const int i = env0 + lane;
        if (wave == 2 && lane < R) noise[(k + 1) & 1][lane] = gaussian_noise(sseed + a.sample_stride, i, A, 0);
        if (wave > 1 || lane >= ne) continue;
        // wavefronts 0 and 1 draw the action; 1 goes on to its log-probability and the rollout row, 0 to the env step
        float av[A];
        const float logp = sample_gaussian(logits + lane * (PA_MAX + 1), w2a + HEAD_LOG_STD(H), A, sseed, i, av, &stdv, noise[k & 1] + lane);
        if (wave == 1) {
            a.r_actions[row + lane] = av[0];
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
        slot.store(a.states, env0 + t);
#pragma unroll
        for (int c = 0; c < IN; ++c) a.obs[(size_t)(env0 + t) * IN + c] = slot.obs(c);
        a.acc.ep_return[env0 + t] = ep_return;
        a.acc.ep_length[env0 + t] = ep_length;
    }
}

// Hidden width 64, as CartPole's: the critic on two wavefronts of its own.  Wavefront 0 carries the envs, in all four lanes of
// one's row of the head, and goes on from the head's sum to the action and the env step.
//   wavefronts 0 .. 3   layer 0           layer 1              0: head, env step; 1: the normal numbers of step k + 1
//              4        rewards of k - 1  critic's head k - 1  log-probability of k - 1
//              5        observations out  sine of the angle
//              6, 7     critic's layer 0  critic's layer 1 ... ...
template <int ACT>
__global__ __launch_bounds__(512, 4) void collect_pendulum16_h64_kernel(CollectArgs a) {
    constexpr int H = 64, IN = pendulum::OBS, R = PR16, T = 512, KB = H / 4, EARLY = 8;
    struct Row { float obs[IN], theta, sine; };
    __shared__ Row rows[R];
    __shared__ float noise[2][R], mean[R], action[R], rew[R], don[R];
    __shared__ float hT[2][H * HT16_LD];
    __shared__ float h2[2][R * (H + 1)];
    __shared__ __align__(16) float w2a[HEAD_LDS(H)];
    __shared__ float w2c[H + 1];
    __shared__ EpisodeBooks::Waiting finished;
    const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t / WAVE), lane = t % WAVE;
    const int env0 = blockIdx.x * R;
    const int nenv = min(R, a.n_envs - env0);
    const int N = a.n_envs;
    const size_t row0 = (size_t)a.t0 * N + env0;   // the first step's rollout row
    const int e = lane >> 2, l = lane & 3;
    stage_head(a.actor_p + IN * H + H + H * H + H, H, 1, true, w2a, t, T);
    for (int i = t; i < H + 1; i += T) w2c[i] = a.critic_p[IN * H + H + H * H + H + i];
    auto input = [&](float (&a0)[1]) {
        const int g = lane >> 4;
        a0[0] = g < IN ? rows[lane & 15].obs[g < IN ? g : 0] : 0.0f;
    };
    if (wave < 4) {
        PendulumSlot slot{};
        if (wave == 0) {
            if (e < nenv) slot.load(a.states, env0 + e);
            if (l == 0) {
#pragma unroll
                for (int c = 0; c < IN; ++c) rows[e].obs[c] = slot.obs(c);
                rows[e].theta = slot.s[3];
            }
        } else if (wave == 1 && lane < R) {
            noise[0][lane] = gaussian_noise(a.sample_seed, env0 + lane, 1, 0);
        }
        Hidden16Operands<H, IN, 1, KB> ops;
        const int c0 = 16 * wave;
        ops.load(a.actor_p, c0, lane);
        __syncthreads();
        HeadRow16<H, 1, PA_MAX> head;
        head.load(w2a, l);
        const float std = exp32(gaussian_log_std(w2a[HEAD_LOG_STD(H)]));
        for (int k = 0; k < a.n_steps; ++k) {
            float a0[1];
            input(a0);
            hidden16_layer0_of<H, IN, ACT, 1, KB>(a0, hT[0], ops, c0, lane);
            __syncthreads();
            floatx4 p[1] = {floatx4{0}};
            hidden16_layer1_steps<H, 0, KB>(hT[0], ops, p, lane);
            hidden16_layer1_end<H, IN, ACT, 1, KB>(p, h2[0], ops, c0, lane);
            __syncthreads();
            if (wave == 0) {
                const float sine = rows[e].sine, z = noise[k & 1][e];
                float mu[1], r, d;
                head.sums(h2[0], e, l, mu);
                const float u = mu[0] + std * z;
                pendulum::step(slot.s, u, sine, r, d);
                if (d > 0.5f) slot.reset(env0 + e, a.reset_seed + (uint64_t)k * a.reset_stride);
                if (l == 0) {
#pragma unroll
                    for (int c = 0; c < IN; ++c) rows[e].obs[c] = slot.obs(c);
                    rows[e].theta = slot.s[3];
                    mean[e] = mu[0];
                    action[e] = u;
                    rew[e] = r;
                    don[e] = d;
                }
            } else if (wave == 1 && lane < R) {
                noise[(k + 1) & 1][lane] = gaussian_noise(a.sample_seed + (uint32_t)(k + 1) * a.sample_stride, env0 + lane, 1, 0);
            }
            __syncthreads();
        }
        if (wave == 0 && l == 0 && e < nenv) {
            slot.store(a.states, env0 + e);
#pragma unroll
            for (int c = 0; c < IN; ++c) a.obs[(size_t)(env0 + e) * IN + c] = slot.obs(c);
        }
    } else if (wave == 4) {
        const bool mine = lane < nenv;
        const int q = lane & (R - 1);
        EpisodeBooks books;
        books.begin(a, env0 + lane, mine);
        __syncthreads();
        HeadRow16<H, 1, 1> head;
        head.load(w2c, l);
        const float log_std = gaussian_log_std(w2a[HEAD_LOG_STD(H)]), std = exp32(log_std);
        float u = 0.0f, mu = 0.0f;
        auto rewards = [&](int k) {
            u = action[q];
            mu = mean[q];
            const size_t at = row0 + (size_t)k * N + lane;
            if (mine) a.r_actions[at] = u;
            books.rewards(a, finished, k, at, rew[q], don[q], lane, mine);
        };
        auto value = [&](int k) {
            float out[1];
            head.sums(h2[1], e, l, out);
            if (l == 0 && e < nenv) a.r_values[row0 + (size_t)k * N + e] = out[0];
        };
        auto logp = [&](int k) {
            if (mine) a.r_logp[row0 + (size_t)k * N + lane] = 0.0f + gaussian_logp(u, mu, log_std, std);
        };
        for (int k = 0; k < a.n_steps; ++k) {
            if (k > 0) rewards(k - 1);
            __syncthreads();
            if (k > 0) value(k - 1);
            __syncthreads();
            if (k > 0) logp(k - 1);
            __syncthreads();
        }
        if (a.n_steps > 0) {
            rewards(a.n_steps - 1);
            value(a.n_steps - 1);
            logp(a.n_steps - 1);
        }
        books.end(a, finished, env0 + lane, lane, mine);
    } else if (wave == 5) {
        __syncthreads();
        for (int k = 0; k < a.n_steps; ++k) {
            const int q = lane & (R - 1);
            const float theta = rows[q].theta;
            if (lane < nenv) {
#pragma unroll
                for (int c = 0; c < IN; ++c) a.r_obs[(row0 + (size_t)k * N + lane) * IN + c] = rows[q].obs[c];
            }
            __syncthreads();
            if (lane < R) rows[lane].sine = sin32(theta);
            __syncthreads();
            __syncthreads();
        }
    } else {
        Hidden16Operands<H, IN, 2, KB> ops;
        const int c0 = 32 * (wave - 6);
        ops.load(a.critic_p, c0, lane);
        __syncthreads();
        for (int k = 0; k < a.n_steps; ++k) {
            float a0[1];
            input(a0);
            hidden16_layer0_of<H, IN, ACT, 2, KB>(a0, hT[1], ops, c0, lane);
            __syncthreads();
            floatx4 p[2] = {floatx4{0}, floatx4{0}};
            hidden16_layer1_steps<H, 0, EARLY>(hT[1], ops, p, lane);
            __syncthreads();
            hidden16_layer1_steps<H, EARLY, KB>(hT[1], ops, p, lane);
            hidden16_layer1_end<H, IN, ACT, 2, KB>(p, h2[1], ops, c0, lane);
            __syncthreads();
        }
    }
}

template <int H, int ACT>
void launch_cartpole16(mrl_ctx *ctx, dim3 grid, const CollectArgs &a, int32_t *side) {
    if constexpr (H == 64) hipLaunchKernelGGL((collect_cartpole16_h64_kernel<ACT>), grid, dim3(512), 0, ctx->stream, a, side);
    else hipLaunchKernelGGL((collect_cartpole16_kernel<H, ACT>), grid, dim3(512), 0, ctx->stream, a, side);
}

template <int H, int ACT>
void launch_pendulum16(mrl_ctx *ctx, dim3 grid, const CollectArgs &a) {
    if constexpr (H == 64) hipLaunchKernelGGL((collect_pendulum16_h64_kernel<ACT>), grid, dim3(512), 0, ctx->stream, a);
    else hipLaunchKernelGGL((collect_pendulum16_kernel<H, ACT>), grid, dim3(512), 0, ctx->stream, a);
}

// the workgroups of `grid` = 16 envs each; side: CartPole's step counters
template <int H, int ACT>
int launch_collect16_t(mrl_ctx *ctx, const mrl_rollout *r, const CollectArgs &a, int32_t *side) {
    const dim3 grid(grid_for(r->n_envs, PR16)), block(LunarLander::THREADS);
    const bool wide = (int)grid.x <= ctx->n_cus;
    if (r->env_id == MRL_ENV_LUNARLANDER && wide)
        hipLaunchKernelGGL((collect16_wide_kernel<LunarLander, H, ACT, false>), grid, dim3(512), 0, ctx->stream, a);
    else if (r->env_id == MRL_ENV_LUNARLANDER)
        hipLaunchKernelGGL((collect16_kernel<LunarLander, H, ACT, false>), grid, block, 0, ctx->stream, a);
    else if (r->env_id == MRL_ENV_LUNARLANDER_CONTINUOUS && wide)
        hipLaunchKernelGGL((collect16_wide_kernel<LunarLanderContinuous, H, ACT, true>), grid, dim3(512), 0, ctx->stream, a);
    else if (r->env_id == MRL_ENV_LUNARLANDER_CONTINUOUS)
        hipLaunchKernelGGL((collect16_kernel<LunarLanderContinuous, H, ACT, true>), grid, block, 0, ctx->stream, a);
    else if (r->env_id == MRL_ENV_CARTPOLE)
        launch_cartpole16<H, ACT>(ctx, grid, a, side);
    else
        launch_pendulum16<H, ACT>(ctx, grid, a);
    MRL_CHECK_LAUNCH();
    return MRL_OK;
}

}  // namespace mrl
