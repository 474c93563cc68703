// What a fused collection step leaves beside the envs' rows, written by a wavefront that the step does not wait for.
#pragma once
#include "mrl_device.hpp"
#include "mlp_tile16.hpp"
#include "policy_sample.hpp"
#include "env_block.hpp"
#include "collect_args.hpp"

namespace mrl {

// Reward and done flag of a step into the rollout, and the episode sums, a lane per env of one wavefront.  Finished episodes wait
// in LDS for the workgroup's turn, every sixteenth step, or until some dozens are there: their places in the list come from one
// counter of the whole chip, at which a request per step and workgroup were what a step of 4096 envs waited for.  So the list is
// in the order in which episodes end to within the sixteen steps and what the workgroups are apart (CartPole, H = 64, us per step
// at 1024 / 4096 envs, kept until dozens are there : with turns: 1.41 / 1.53 : 1.43 / 1.55; an episode stood behind others that
// ended up to 68 steps after it, now 15).  (All lanes of the wavefront make the calls.)
struct EpisodeBooks {
    static constexpr int R = PR16, EVERY = 16;
    struct Waiting { float ret[WAVE], len[WAVE]; };
    float ep_return = 0.0f, ep_length = 0.0f;
    int waiting = 0;
    MRL_DEV void begin(const CollectArgs &a, int env, bool mine) {
        if (mine) {
            ep_return = a.acc.ep_return[env];
            ep_length = a.acc.ep_length[env];
        }
    }
    MRL_DEV void list(const CollectArgs &a, const Waiting &w, int lane) {
        int first = 0;
        if (lane == 0) first = atomicAdd(a.acc.done_count, waiting);
        first = __builtin_amdgcn_readfirstlane(first);
        if (lane < waiting && first + lane < a.acc.done_cap) {
            a.acc.done_returns[first + lane] = w.ret[lane];
            a.acc.done_lengths[first + lane] = w.len[lane];
        }
        waiting = 0;
    }
    MRL_DEV void rewards(const CollectArgs &a, Waiting &w, int k, size_t at, float r, float d, int lane, bool mine) {
        if (mine) {
            a.r_rewards[at] = r;
            a.r_dones[at] = d;
        }
        ep_return = ep_return + r;
        ep_length = ep_length + 1.0f;
        const bool finished = mine && d > 0.5f;
        const unsigned long long all = __ballot(finished);
        const bool turn = ((k + (int)blockIdx.x) & (EVERY - 1)) == 0;
        if (finished) {
            const int i = waiting + __popcll(all & ((1ull << lane) - 1));
            w.ret[i] = ep_return;
            w.len[i] = ep_length;
        }
        ep_return = finished ? 0.0f : ep_return;
        ep_length = finished ? 0.0f : ep_length;
        waiting += __popcll(all);
        if (waiting > (turn ? 0 : WAVE - R)) list(a, w, lane);
    }
    MRL_DEV void end(const CollectArgs &a, const Waiting &w, int env, int lane, bool mine) {
        if (waiting > 0) list(a, w, lane);
        if (mine) {
            a.acc.ep_return[env] = ep_return;
            a.acc.ep_length[env] = ep_length;
        }
    }
};

// What the steps of a Gaussian policy hand to the wavefront that writes the rollout rows; step k's at [k & 1], the normal numbers
// there a step ahead.  std, log_std: the policy does not change during a launch.
template <int AW>
struct GaussBooks {
    static constexpr int R = PR16;
    float noise[2][R * AW], mean[2][R * AW], act[2][R * AW], rew[2][R], don[2][R], vals[2][R];
    float log_std[AW], std[AW];
    EpisodeBooks::Waiting finished;

    MRL_DEV void make_noise(const CollectArgs &a, int k, int env0, int i) {
        noise[k & 1][i] = gaussian_noise(a.sample_seed + (uint32_t)k * a.sample_stride, env0 + i / AW, AW, i % AW);
    }
    // ahead of the first step, all threads of the workgroup (at least R * AW); head: the actor's in global memory, log_std last
    MRL_DEV void begin(const CollectArgs &a, const float *log_std_p, int env0, int t) {
        if (t < R * AW) make_noise(a, 0, env0, t);
        if (t < AW) {
            log_std[t] = gaussian_log_std(log_std_p[t]);
            std[t] = exp32(log_std[t]);
        }
    }
    // component i % AW of env i / AW, given its mean
    MRL_DEV void draw(int k, int i, float mu) {
        mean[k & 1][i] = mu;
        act[k & 1][i] = mu + std[i % AW] * noise[k & 1][i];
    }
    // step k into the rollout, by one wavefront
    MRL_DEV void book(EpisodeBooks &b, const CollectArgs &a, int k, int env0, int lane, bool mine) {
        const int q = k & 1, e = lane & (R - 1);
        const size_t at = (size_t)(a.t0 + k) * a.n_envs + env0 + lane;
        if (mine) {
            float logp = 0.0f;
#pragma unroll
            for (int j = 0; j < AW; ++j) {
                const float u = act[q][e * AW + j];
                logp = logp + gaussian_logp(u, mean[q][e * AW + j], log_std[j], std[j]);
                a.r_actions[at * AW + j] = u;
            }
            a.r_logp[at] = logp;
            a.r_values[at] = vals[q][e];
        }
        b.rewards(a, finished, k, at, rew[q][e], don[q][e], lane, mine);
    }
};

}  // namespace mrl
