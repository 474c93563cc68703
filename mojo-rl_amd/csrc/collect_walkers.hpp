// Fused collection kernels of the continuous-control envs beyond the classic ones (BipedalWalker,
// HalfCheetah planar, CarRacingV2, HopperPlanar, Walker2dPlanar) with the agents' Gaussian nets (hidden width H = 64, 128 or 256): many rollout
// steps of a block's 16 envs in ONE launch, like the kernels of mrl_collect.hip.  The env rows (CarRacing: the 40
// floats in front of the track) stay in LDS from the first step to the last; per step and block
//   policy   the actor  OBS -> H -> H -> A  on wavefronts 0 .. 3 and the critic  OBS -> H -> H -> 1
//            on four others, on the fp32 matrix cores (the 16-row tiles of mlp_tile16.hpp, H / 4 columns
//            per wavefront, weights streamed from L2), heads out of LDS.  The walkers: only the actor runs
//            ahead of the env step; the critic, whose value is only stored, runs beside the one-lane-per-
//            body solver on wavefronts 2, 3, 6 and 7 (the two SIMDs that the solver's wavefronts 0 and 1
//            do not use).  CarRacing, whose env step takes every wavefront: both nets side by side
//            (critic on wavefronts 4 .. 7) ahead of it;
//   sample   one lane per (env, action component): every component has a Philox stream of its own (all but
//            CarRacing: the normal numbers a step ahead, beside the actor);
//   env step BipedalWalker: the workgroup-level step of env_block.hpp (contact detection on every
//            wavefront, solver with one lane per body on wavefronts 0 and 1, lidar rays on every
//            wavefront, wave-cooperative resets); HalfCheetah: one lane per body on wavefronts 0 and 1
//            (env_cheetah_lanes.hpp); CarRacing: a wavefront per env, two rounds of eight (env_car.hpp);
//            the tile tables stay in global memory and are staged through LDS every step (16 x 12 KB do
//            not fit beside the rest); HopperPlanar / Walker2dPlanar: one lane per env on wavefront 0
//            (Float64, env_planar.hpp), the critic beside it as for the walkers, at width 256 on the six
//            wavefronts of the other three SIMDs;
//   rollout row t of obs, action, log-prob, value, reward, done and the episode sums written on the way (all but
//            CarRacing: a step later, by a wavefront that has the time beside the actor).
// With these envs the step is 70 - 80 % env step, a chain of one or two wavefronts' instructions: what the
// fusion buys is the launch gaps, the observation / action round trip through HBM, the staging of the rows
// in and out of LDS every step, and a policy forward of a 16-row tile on one CU.
//
// It gives what n_steps calls of mrl_rollout_step give (same per-env streams: seeds are affine in
// the step number), except that the finished-episode list is appended in the order in which blocks
// get there, every sixteen steps (CarRacing: every step), rather than step by step.
#pragma once
#include <type_traits>
#include "mrl_host.hpp"
#include "mrl_device.hpp"
#include "mlp_tile.hpp"
#include "mlp_tile16.hpp"
#include "policy_sample.hpp"
#include "env_block.hpp"
#include "env_cheetah_lanes.hpp"
#include "env_car.hpp"
#include "env_planar.hpp"
#include "collect_books.hpp"

namespace mrl {

// HalfCheetah's traits with the block shape of this kernel
struct HalfCheetah16 : HalfCheetah {
    static constexpr int EPB = 16, THREADS = 512;
};

template <int A, int B>
constexpr int wmax() { return A > B ? A : B; }

// The policy half of a step, by all 512 threads: observation tile from `obs_at(row, column)` (also out to
// rollout row t), actor on wavefronts 0 .. 3 and critic on 4 .. 7 (tiles = 2 * H * HT16_LD floats of LDS),
// Gaussian sampling on one lane per (env, action component) -- the log-probability is the sum of the
// components' terms in component order --, rollout row t of action, log-prob and value.  Leaves the
// actions in act[env][AW]; ends with the block in step (everything above complete).
template <int H, int IN, int AW, int ACT, class ObsAt>
MRL_DEV void policy16_gauss(const CollectArgs &a, ObsAt obs_at, int tid, int ne, int A, int zero, size_t row,
                            uint32_t sseed, int env0, float *xs, float *tiles, const float *w2a, const float *w2c,
                            float *logits, float *vals, float *act, float *part) {
    constexpr int R = PR16, T = 512, KBA = 8, NT = H / 64;
    const int wave = tid / WAVE, lane = tid % WAVE;
    const int net = wave >> 2;                           // 0: actor, 1: critic
    {
        const float *p = (net ? a.critic_p : a.actor_p) + zero;
        float *tile = tiles + net * (H * HT16_LD);
        Hidden16Operands<H, IN, NT, KBA> ops;
        ops.load(p, 16 * NT * (wave & 3), lane);
        stage_observations<IN, T>(xs, a.r_obs + row * IN, ne, tid, obs_at);
        __syncthreads();
        BlockSync bs;
        hidden_stack16<H, IN, ACT, NT, KBA, true>(p, xs, tile, tile, ops, 16 * NT * (wave & 3), lane, bs);
        if (net == 0) head16<H>(w2a, A, tile, logits, PA_MAX + 1, tid, T / 2);
        else head16_value<H>(w2c, tile, vals, tid - T / 2, T / 2);
        __syncthreads();   // means and values complete; the tiles are dead from here on
    }
    for (int e = tid; e < ne * A; e += T) {
        const int r = e / A, j = e - r * A;
        float av;
        part[r * PA_MAX + j] = sample_gaussian_part(logits + r * (PA_MAX + 1) + j, w2a + HEAD_LOG_STD(H) + j, 1, A, j,
                                                    sseed, env0 + r, &av);
        act[r * AW + j] = av;
        a.r_actions[row * AW + e] = av;
    }
    if (tid < ne) a.r_values[row + tid] = vals[tid];
    __syncthreads();
    if (tid < ne) {
        float logp = 0.0f;
        for (int j = 0; j < A; ++j) logp = logp + part[tid * PA_MAX + j];
        a.r_logp[row + tid] = logp;
    }
}

// The actor's half of policy16_gauss by wavefronts 0 .. 3 alone (the observation tile xs is complete, every
// thread of the four passes its tid): hidden stack on `tile`, the draw from the normal numbers in `b`, which takes the
// actions.  The four wavefronts meet at `sync`, five rounds per call.
// KB = H / 4: the weights are in `ops` already, for the whole launch.
template <int H, int IN, int AW, int ACT, int KB>
MRL_DEV void actor16_gauss(const CollectArgs &a, int tid, int zero, int k, const float *xs, float *tile, const float *w2a,
                           float *logits, GaussBooks<AW> &b, Hidden16Operands<H, IN, H / 64, KB> &ops, WaveGroupSync &sync) {
    constexpr int TA = 4 * WAVE, NT = H / 64;
    const int wave = tid / WAVE, lane = tid % WAVE;
    const float *p = a.actor_p + zero;
    if (4 * KB < H) ops.load(p, 16 * NT * wave, lane);
    hidden_stack16<H, IN, ACT, NT, KB, true>(p, xs, tile, tile, ops, 16 * NT * wave, lane, sync);
    head16<H>(w2a, AW, tile, logits, PA_MAX + 1, tid, TA);
    sync();   // means complete
    if (tid < PR16 * AW) b.draw(k, tid, logits[tid / AW * (PA_MAX + 1) + tid % AW]);
    sync();   // actions complete
}
// What wavefronts 4 .. 7 do beside it: the normal numbers of step k + 1 (4, 6) and the rollout row of step k - 1 (5).  (The
// draws took 2.5 thousand cycles of a step between the head and the env step, the episode sums in global memory 1 to 2
// thousand behind it.  us per step, 4096 envs, H = 64 / 256, in line : here:
// Hopper 7.65 / 19.4 : 6.41 / 19.0, Walker2d 11.3 / 20.4 : 9.85 / 19.3, BipedalWalker 27.7 / 33.4 : 26.1 / 31.7, HalfCheetah
// 40.7 / 45.8 : 39.2 / 44.2.)
template <int AW>
MRL_DEV void beside_actor16(const CollectArgs &a, int wave, int lane, int k, int env0, int ne, GaussBooks<AW> &b, EpisodeBooks &books) {
    static_assert(PR16 * AW <= 2 * WAVE, "a lane per env and component");
    if (wave == 5) {
        if (k > 0) b.book(books, a, k - 1, env0, lane, lane < ne);
    } else if (wave != 7) {
        const int i = (wave == 4 ? 0 : WAVE) + lane;
        if (i < PR16 * AW) b.make_noise(a, k + 1, env0, i);
    }
}
constexpr unsigned ACTOR16_ROUNDS = 5, CRITIC16_ROUNDS = 3;

// The critic's half by wavefronts 2, 3, 6 and 7 (the two SIMDs that do not host wavefronts 0 and 1), on a
// barrier of their own: values of the block's rows into vals.
template <int H, int IN, int ACT>
MRL_DEV void critic16_side(const CollectArgs &a, int zero, int k, int tid, const float *xs, float *tile, const float *w2c,
                           float *vals, unsigned *sync_word, unsigned *failed) {
    constexpr int KBA = 8, NT = H / 64;
    const int wave = tid / WAVE, lane = tid % WAVE;
    if (!(wave & 2)) return;
    const int g = (wave & 1) + ((wave >> 2) << 1);   // 0 .. 3
    const float *p = a.critic_p + zero;
    WaveGroupSync sync{sync_word, (unsigned)k * CRITIC16_ROUNDS * 4u, 4u, failed, a.spin_limit};
    Hidden16Operands<H, IN, NT, KBA> ops;
    ops.load(p, 16 * NT * g, lane);
    hidden_stack16<H, IN, ACT, NT, KBA, true>(p, xs, tile, tile, ops, 16 * NT * g, lane, sync);
    head16_value<H>(w2c, tile, vals, g * WAVE + lane, 4 * WAVE);
}

// The same at hidden width 256 where only wavefront 0 has the env step: on six wavefronts, 1 to 3 and 5 to 7, of the other
// three SIMDs (1, 2, 1 and 4, 4, 4 column tiles).  On two SIMDs the critic is 24 thousand cycles beside a step of 16.  us per
// step, two SIMDs : three: Hopper 18.2 : 16.0 (256 envs), 19.0 : 17.1 (4096), Walker2d 18.6 : 16.2, 19.3 : 17.4; at width 128,
// where the step is the longer one or nearly, 10.4 : 10.0 and 12.4 : 12.7, at width 64 6.4 : 6.6 and 9.8 : 9.8.
template <int H, int IN, int ACT>
MRL_DEV void critic16_wide(const CollectArgs &a, int zero, int k, int wave, int lane, const float *xs, float *tile, const float *w2c,
                           float *vals, unsigned *sync_word, unsigned *failed) {
    static_assert(H == 256, "sixteen column tiles");
    constexpr unsigned CW = 6;
    const float *p = a.critic_p + zero;
    auto share = [&](auto tiles, int m, int c0) {
        constexpr int NT = decltype(tiles)::value;
        WaveGroupSync sync{sync_word, (unsigned)k * CRITIC16_ROUNDS * CW, CW, failed, a.spin_limit};
        Hidden16Operands<H, IN, NT, 8> ops;
        ops.load(p, c0, lane);
        hidden_stack16<H, IN, ACT, NT, 8, true>(p, xs, tile, tile, ops, c0, lane, sync);
        head16_value<H>(w2c, tile, vals, m * WAVE + lane, CW * WAVE);
    };
    if (wave > 4) share(std::integral_constant<int, 4>{}, wave - 5, 64 * (wave - 5));
    else if (wave == 2) share(std::integral_constant<int, 2>{}, 4, 208);
    else if (wave < 4) share(std::integral_constant<int, 1>{}, wave == 1 ? 3 : 5, wave == 1 ? 192 : 240);
}

template <class E, int H, int ACT, bool LANES>
__global__ __launch_bounds__(512) void collect_walker_kernel(CollectArgs a) {
    using S = Stage<E>;
    constexpr int IN = E::OBS, AW = E::ACT_W, R = PR16, T = 512;
    static_assert(E::EPB == R && E::THREADS == T && IN <= PIN_MAX && AW <= PA_MAX, "16 envs per workgroup of eight wavefronts");
    __shared__ float rows[R * S::STRIDE];
    __shared__ float xs[R * XS_LD];
    __shared__ __align__(16) float w2a[HEAD_LDS(H)];
    __shared__ float w2c[H + 1];                    // the critic's head: column of H weights, then the bias
    __shared__ float logits[R * (PA_MAX + 1)];
    __shared__ GaussBooks<AW> b;
    __shared__ float shapes[E::NSHAPE];
    __shared__ unsigned long long was_reset;
    __shared__ unsigned sync_actor, sync_critic, sync_failed;   // barriers of the actor's and the critic's wavefronts
    // the two activation tiles and the env step's scratch (contact lists) are never live together
    constexpr int LIST_F = detect_list_floats<E>() + 1;
    constexpr int ENV_F = R * S::CSTRIDE + LIST_F + detect_count_ints<E>();
    // the critic's tile: above the actor's and above the solver's contact scratch, below the merged counts
    constexpr int CRITIC_OFF = wmax<H * HT16_LD, R * S::CSTRIDE>();
    __shared__ float overlay[wmax<CRITIC_OFF + H * HT16_LD, ENV_F>()];
    static_assert(LANES || CRITIC_OFF + H * HT16_LD <= R * S::CSTRIDE + LIST_F, "the critic's tile lies over spent contact lists only");
    float *cts = overlay, *dlist = cts + R * S::CSTRIDE;
    int *dcount = reinterpret_cast<int *>(dlist + LIST_F);

    const int t = threadIdx.x;
    const int env0 = blockIdx.x * R;
    const int nenv = min(R, a.n_envs - env0);
    const int N = a.n_envs;
    float *gbase = a.states + (size_t)env0 * E::STATE;

    S::in(rows, gbase, nenv, t);
    for (int i = t; i < E::NSHAPE; i += T) shapes[i] = a.shapes[i];
    stage_head(a.actor_p + IN * H + H + H * H + H, H, a.A, true, w2a, t, T);
    for (int i = t; i < H + 1; i += T) w2c[i] = a.critic_p[IN * H + H + H * H + H + i];
    b.begin(a, a.actor_p + IN * H + H + H * H + H + (H + 1) * AW, env0, t);
    EpisodeBooks books;   // wavefront 5's
    books.begin(a, env0 + t - 5 * WAVE, t >= 5 * WAVE && t - 5 * WAVE < nenv);
    if (t == 0) {
        was_reset = 0;
        sync_actor = 0;
        sync_critic = 0;
        sync_failed = 0;
    }
    __syncthreads();

    for (int k = 0; k < a.n_steps; ++k) {
        // nothing but the rows is carried from one step to the next (see collect16_kernel)
        int tid = t, ne = __builtin_amdgcn_readfirstlane(nenv), zero = 0;
        asm volatile("" : "+v"(tid), "+s"(zero), "+s"(ne) : : "memory");
        const int now = k & 1;
        const size_t row = (size_t)(a.t0 + k) * N + env0;   // this block's slice of rollout row t
        const uint64_t rseed = a.reset_seed + (uint64_t)k * a.reset_stride;
        const int wave = tid / WAVE, lane = tid % WAVE;
        // The env step keeps wavefronts 0 and 1 busy for most of the step (the solver with one lane per body)
        // and the others for little or nothing: only the actor goes ahead of it (wavefronts 0 .. 3, one per
        // SIMD); the critic, whose value is only stored, runs beside the solver on wavefronts 2, 3, 6 and 7 --
        // the two SIMDs that do not host wavefronts 0 and 1.  Both groups meet at bounded barriers of their
        // own, rebuilt every step from the step number.
        stage_observations<IN, T>(xs, a.r_obs + row * IN, ne, tid, [&](int r, int c) { return rows[r * S::STRIDE + c]; });
        __syncthreads();
        if (wave < 4) {
            WaveGroupSync actor_sync{&sync_actor, (unsigned)k * ACTOR16_ROUNDS * 4u, 4u, &sync_failed, a.spin_limit};
            Hidden16Operands<H, IN, H / 64, 8> ops;
            actor16_gauss<H, IN, AW, ACT>(a, tid, zero, k, xs, overlay, w2a, logits, b, ops, actor_sync);
        } else {
            beside_actor16<AW>(a, wave, lane, k, env0, ne, b, books);
        }
        float *critic_tile = overlay + CRITIC_OFF;   // (above the env step's contact scratch cts)
        // ---- env step with auto-reset
        if constexpr (!LANES) {
            // (the critic's tile lies over contact lists that are spent by the time the solver runs)
            auto side = [&](int th) {
                critic16_side<H, IN, ACT>(a, zero, k, th, xs, critic_tile, w2c, b.vals[now], &sync_critic, &sync_failed);
            };
            phys_step_block<E, true>(rows, cts, shapes, dlist, dcount, &was_reset, b.act[now], b.rew[now], b.don[now], env0, ne,
                                     rseed, Accounting{}, tid, side);
        } else {
            // HalfCheetah: eight lanes per env, eight envs per wavefront, on wavefronts 0 and 1; a row
            // whose wiring is not HalfCheetah's own is stepped by lane 0 of its group in the one-lane form
            if (wave < 2) {
                const int slot = wave * 8 + (lane >> 3), l = lane & 7;
                const bool live = slot < ne;
                float *rowp = rows + slot * S::STRIDE;
                const int env = env0 + (live ? slot : 0);
                const float *ap = b.act[now] + (live ? slot : 0) * AW;
                const bool ok = live && hc::lanes_row_ok(rowp, shapes);
                float r = 0.0f, d = 0.0f;
                if (ok) hc::step_lanes(rowp, shapes, ap, lane, r, d);
                else if (live && l == 0) hc::step_row(rowp, cts + slot * S::CSTRIDE, shapes, env, ap, r, d);
                if (live && l == 0) {
                    b.rew[now][slot] = r;
                    b.don[now][slot] = d;
                    if (d > 0.5f) E::reset(rowp, rseed, env);
                }
            } else {
                critic16_side<H, IN, ACT>(a, zero, k, tid, xs, critic_tile, w2c, b.vals[now], &sync_critic, &sync_failed);
            }
        }
        __syncthreads();   // env step done: the rows hold the next observation
        // a wait that gave up: the block's results are void from here on; leave the loop and end normally
        if (sync_failed != 0u) break;
    }
    if (sync_failed != 0u) {
        // a wait gave up: the step in progress ran on data that was never produced; the block's rows and
        // observations are not stored and keep the values from before the launch
        if (t == 0) *a.sync_error = 1;
        return;
    }
    if (t / WAVE == 5) {
        const int lane = t % WAVE;
        if (a.n_steps > 0) b.book(books, a, a.n_steps - 1, env0, lane, lane < nenv);
        books.end(a, b.finished, env0 + lane, lane, lane < nenv);
    }

    for (int i = t; i < nenv * E::OBS; i += T) {
        const int r = i / E::OBS, c = i - r * E::OBS;
        a.obs[(size_t)env0 * E::OBS + i] = rows[r * S::STRIDE + c];
    }
    S::out(rows, gbase, nenv, t, 0, E::STATE);
}

// CarRacingV2: the rows stay in global memory (12 KB each, nearly all of it the track); the block keeps the
// 40 floats in front of the track -- observation, hull, wheels, controls, metadata -- of its 16 envs in LDS
// over the whole launch.  Env step: a wavefront per env in two rounds of eight; each wavefront stages its
// env's tile table through LDS (over the activation tiles, which are dead by then), steps, accounts, and
// rebuilds the env when it finished (one lane walks the new track: only this block waits for it).
template <int H, int ACT>
__global__ __launch_bounds__(512) void collect_car_kernel(CollectArgs a) {
    constexpr int IN = cr::OBS, AW = cr::ACT, R = PR16, T = 512, HEAD = cr::TRACK;
    static_assert(IN <= PIN_MAX && AW <= PA_MAX && cr::TABLE % 4 == 0, "tile limits");
    __shared__ float heads[R * (HEAD + 1)];
    __shared__ float xs[R * XS_LD];
    __shared__ __align__(16) float w2a[HEAD_LDS(H)];
    __shared__ float w2c[H + 1];
    __shared__ float logits[R * (PA_MAX + 1)];
    __shared__ float vals[R];
    __shared__ float act[R * PA_MAX];
    __shared__ float part[R * PA_MAX];
    __shared__ __align__(16) float overlay[wmax<2 * H * HT16_LD, 8 * cr::TABLE>()];

    const int t = threadIdx.x;
    const int env0 = blockIdx.x * R;
    const int nenv = min(R, a.n_envs - env0);
    const int N = a.n_envs;
    for (int i = t; i < nenv * HEAD; i += T) {
        const int r = i / HEAD, c = i - r * HEAD;
        heads[r * (HEAD + 1) + c] = a.states[(size_t)(env0 + r) * cr::STATE + c];
    }
    stage_head(a.actor_p + IN * H + H + H * H + H, H, a.A, true, w2a, t, T);
    for (int i = t; i < H + 1; i += T) w2c[i] = a.critic_p[IN * H + H + H * H + H + i];
    __syncthreads();

    for (int k = 0; k < a.n_steps; ++k) {
        int tid = t, ne = __builtin_amdgcn_readfirstlane(nenv), A = __builtin_amdgcn_readfirstlane(a.A), zero = 0;
        asm volatile("" : "+v"(tid), "+s"(zero), "+s"(ne), "+s"(A) : : "memory");
        const size_t row = (size_t)(a.t0 + k) * N + env0;
        const uint32_t sseed = a.sample_seed + (uint32_t)k * a.sample_stride;
        const uint64_t rseed = a.reset_seed + (uint64_t)k * a.reset_stride;
        const int wave = tid / WAVE, sub = tid % WAVE;
        policy16_gauss<H, IN, AW, ACT>(a, [&](int r, int c) { return heads[r * (HEAD + 1) + c]; }, tid, ne, A, zero, row, sseed,
                                    env0, xs, overlay, w2a, w2c, logits, vals, act, part);
        Accounting acc = a.acc;
        acc.r_rewards = a.r_rewards + (size_t)(a.t0 + k) * N;
        acc.r_dones = a.r_dones + (size_t)(a.t0 + k) * N;
        acc = acc.at(env0);
        __syncthreads();   // the sampling's reads of the means are done before the tables go over the tiles
#pragma unroll 1
        for (int round = 0; round < 2; ++round) {
            const int slot = round * 8 + wave;
            if (slot < ne) {
                const int env = env0 + slot;
                float *head = heads + slot * (HEAD + 1);
                float *grow = a.states + (size_t)env * cr::STATE;
                float r, d, ob[cr::OBS];
                cr::step_wave<true>(head, grow, overlay + wave * cr::TABLE, act + slot * AW, sub, r, d, ob,
                                    a.car_trait_form != 0);
                if (sub == 0) account(acc, slot, r, d);
                if (d > 0.5f) {
                    float sx, sy, sa;
                    const int nt = cr::reset_group<cr::STEP_LANES>(grow, cr::combined_seed(rseed, env), sub, sx, sy, sa);
                    if (sub < HEAD) {
                        float v = 0.0f;
                        if (sub == 0 || sub == cr::HULL + cr::H_X) v = sx;
                        else if (sub == 1 || sub == cr::HULL + cr::H_Y) v = sy;
                        else if (sub == 2 || sub == cr::HULL + cr::H_ANGLE) v = sa;
                        else if (sub == cr::META + cr::M_NUM_TILES) v = (float)nt;
                        head[sub] = v;
                    }
                    // the new track is read back by this wavefront at its next step: nothing older may
                    // linger in the vector cache
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
                }
            }
        }
        __syncthreads();   // env step done: the heads hold the next observation
    }

    for (int i = t; i < nenv * HEAD; i += T) {
        const int r = i / HEAD, c = i - r * HEAD;
        a.states[(size_t)(env0 + r) * cr::STATE + c] = heads[r * (HEAD + 1) + c];
    }
    for (int i = t; i < nenv * IN; i += T) {
        const int r = i / IN, c = i - r * IN;
        a.obs[(size_t)env0 * IN + i] = heads[r * (HEAD + 1) + c];
    }
}

// HopperPlanar / Walker2dPlanar (env_planar.hpp): the rows (248 / 392 bytes, Float64 state behind the fp32
// observation) stay in LDS over the whole launch; the actor runs on wavefronts 0 .. 3, beside it the next step's normal
// numbers (wavefronts 4 and 6) and the last step's rollout row and episode sums (5), then lanes 0 .. 15 of
// wavefront 0 step one env each (Float64, state in registers for the four sub-steps) and rebuild
// finished rows in place, while the critic runs beside them on wavefronts 2, 3, 6 and 7, at width 256 on 1 to 3 and 5 to 7.
template <class M, int H, int ACT>
__global__ __launch_bounds__(512) void collect_planar_kernel(CollectArgs a) {
    // Widths up to which the actor's weights stay in registers.  Hopper's two workgroups a CU want no more than 128 of them.
    // us per step, 4096 envs, loaded every step : held: Hopper, width 64, 6.41 : 6.32, Walker2d, 64 / 128, 9.85 / 12.4 : 9.61 / 11.8.
    constexpr int HELD = M::STATE == planar::Hopper::STATE ? 64 : 128;
    constexpr int IN = M::OBS, AW = M::ACT, R = PR16, T = 512;
    static_assert(IN <= PIN_MAX && AW <= PA_MAX && M::STATE % 2 == 0, "tile limits; rows are whole doubles");
    __shared__ __align__(16) float rows[R * M::STATE];
    __shared__ float xs[R * XS_LD];
    __shared__ __align__(16) float w2a[HEAD_LDS(H)];
    __shared__ float w2c[H + 1];
    __shared__ float logits[R * (PA_MAX + 1)];
    __shared__ GaussBooks<AW> b;
    __shared__ unsigned sync_actor, sync_critic, sync_failed;
    __shared__ __align__(16) float tiles[2 * H * HT16_LD];

    const int t = threadIdx.x;
    const int env0 = blockIdx.x * R;
    const int nenv = min(R, a.n_envs - env0);
    const int N = a.n_envs;
    float2 *g2 = reinterpret_cast<float2 *>(a.states + (size_t)env0 * M::STATE);
    float2 *l2 = reinterpret_cast<float2 *>(rows);
    for (int i = t; i < nenv * (M::STATE / 2); i += T) l2[i] = g2[i];
    stage_head(a.actor_p + IN * H + H + H * H + H, H, a.A, true, w2a, t, T);
    for (int i = t; i < H + 1; i += T) w2c[i] = a.critic_p[IN * H + H + H * H + H + i];
    b.begin(a, a.actor_p + IN * H + H + H * H + H + (H + 1) * AW, env0, t);
    constexpr int KB = H <= HELD ? H / 4 : 8;   // k-steps of the actor's layer 1 held (all of them, or the next block)
    Hidden16Operands<H, IN, H / 64, KB> ops;
    if (4 * KB == H && t < 4 * WAVE) ops.load(a.actor_p, 16 * (H / 64) * (t / WAVE), t % WAVE);
    EpisodeBooks books;   // wavefront 5's
    books.begin(a, env0 + t - 5 * WAVE, t >= 5 * WAVE && t - 5 * WAVE < nenv);
    if (t == 0) {
        sync_actor = 0;
        sync_critic = 0;
        sync_failed = 0;
    }
    __syncthreads();

    for (int k = 0; k < a.n_steps; ++k) {
        // nothing but the rows is carried from one step to the next (see collect16_kernel)
        int tid = t, ne = __builtin_amdgcn_readfirstlane(nenv), zero = 0;
        asm volatile("" : "+v"(tid), "+s"(zero), "+s"(ne) : : "memory");
        const int now = k & 1;
        const size_t row = (size_t)(a.t0 + k) * N + env0;
        const uint64_t rseed = a.reset_seed + (uint64_t)k * a.reset_stride;
        const int wave = tid / WAVE, lane = tid % WAVE;
        stage_observations<IN, T>(xs, a.r_obs + row * IN, ne, tid, [&](int r, int c) { return rows[r * M::STATE + c]; });
        __syncthreads();
        if (wave < 4) {
            WaveGroupSync actor_sync{&sync_actor, (unsigned)k * ACTOR16_ROUNDS * 4u, 4u, &sync_failed, a.spin_limit};
            actor16_gauss<H, IN, AW, ACT>(a, tid, zero, k, xs, tiles, w2a, logits, b, ops, actor_sync);
        } else {
            beside_actor16<AW>(a, wave, lane, k, env0, ne, b, books);
        }
        if (wave == 0) {
            if (lane < ne) {
                float *rowp = rows + lane * M::STATE;
                planar::State<M> s;
                s.load(rowp);
                float r, d;
                planar::step<M>(s, b.act[now] + lane * AW, r, d);
                b.rew[now][lane] = r;
                b.don[now][lane] = d;
                if (d > 0.5f) planar::reset<M>(s, planar::combined_seed(rseed, env0 + lane));
                s.store(rowp);
            }
        } else {
            float *tile = tiles + H * HT16_LD;
            if constexpr (H == 256) critic16_wide<H, IN, ACT>(a, zero, k, wave, lane, xs, tile, w2c, b.vals[now], &sync_critic, &sync_failed);
            else critic16_side<H, IN, ACT>(a, zero, k, tid, xs, tile, w2c, b.vals[now], &sync_critic, &sync_failed);
        }
        __syncthreads();   // env step done: the rows hold the next observation
        if (sync_failed != 0u) break;
    }
    if (sync_failed != 0u) {
        // a wait gave up: the block's rows and observations keep the values from before the launch
        if (t == 0) *a.sync_error = 1;
        return;
    }
    if (t / WAVE == 5) {
        const int lane = t % WAVE;
        if (a.n_steps > 0) b.book(books, a, a.n_steps - 1, env0, lane, lane < nenv);
        books.end(a, b.finished, env0 + lane, lane, lane < nenv);
    }
    for (int i = t; i < nenv * IN; i += T) {
        const int r = i / IN, c = i - r * IN;
        a.obs[(size_t)env0 * IN + i] = rows[r * M::STATE + c];
    }
    for (int i = t; i < nenv * (M::STATE / 2); i += T) g2[i] = l2[i];
}

template <int H, int ACT>
int launch_collect_walker_t(mrl_ctx *ctx, const mrl_rollout *r, const CollectArgs &args) {
    CollectArgs a = args;
    const dim3 grid(grid_for(r->n_envs, PR16)), block(512);
    if (r->env_id == MRL_ENV_BIPEDAL) {
        a.shapes = ctx->bw_shapes;
        hipLaunchKernelGGL((collect_walker_kernel<BipedalWalker, H, ACT, false>), grid, block, 0, ctx->stream, a);
    } else if (r->env_id == MRL_ENV_CARRACING) {
        hipLaunchKernelGGL((collect_car_kernel<H, ACT>), grid, block, 0, ctx->stream, a);
    } else if (r->env_id == MRL_ENV_HOPPER_PLANAR) {
        hipLaunchKernelGGL((collect_planar_kernel<planar::Hopper, H, ACT>), grid, block, 0, ctx->stream, a);
    } else if (r->env_id == MRL_ENV_WALKER2D_PLANAR) {
        hipLaunchKernelGGL((collect_planar_kernel<planar::Walker2d, H, ACT>), grid, block, 0, ctx->stream, a);
    } else {
        a.shapes = ctx->hc_shapes;
        hipLaunchKernelGGL((collect_walker_kernel<HalfCheetah16, H, ACT, true>), grid, block, 0, ctx->stream, a);
    }
    MRL_CHECK_LAUNCH();
    return MRL_OK;
}

}  // namespace mrl
