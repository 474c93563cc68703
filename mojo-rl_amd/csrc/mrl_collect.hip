// Fused collection: many rollout steps of a block's envs in ONE launch.
//
// Envs do not interact and the policy does not change during a rollout, so a workgroup can take
// its envs through any number of steps on its own: the env rows stay in LDS (registers) from the first step
// to the last (HBM sees them once in and once out per launch, however many steps), the
// observation tile feeds the policy straight from those rows, and the sampled actions reach the
// env step through LDS; rollout row t is written on the way.
// No workgroup waits for another, so there is nothing between two steps but the block's own
// barriers; the launch ends when every block has done its n_steps.
// The kernels: collect16.hpp (LunarLander, CartPole, Pendulum), collect_walkers.hpp (the others); here the entry that picks
// one, or single steps.
//
// It gives what n_steps calls of mrl_rollout_step give (same per-env streams: seeds are affine
// in the step number), except that the finished-episode list is appended, every sixteen steps, in the order in which
// blocks get there rather than step by step.
#include "mrl_host.hpp"
#include "mrl_device.hpp"
#include "mlp_tile.hpp"
#include "policy_sample.hpp"
#include "env_car.hpp"
#include "env_planar.hpp"
#include "collect16.hpp"

namespace mrl {

// compiled in mrl_collect16_h*.hip
extern template int launch_collect16_t<64, 1>(mrl_ctx *, const mrl_rollout *, const CollectArgs &, int32_t *);
extern template int launch_collect16_t<64, 2>(mrl_ctx *, const mrl_rollout *, const CollectArgs &, int32_t *);
extern template int launch_collect16_t<128, 1>(mrl_ctx *, const mrl_rollout *, const CollectArgs &, int32_t *);
extern template int launch_collect16_t<128, 2>(mrl_ctx *, const mrl_rollout *, const CollectArgs &, int32_t *);
extern template int launch_collect16_t<256, 1>(mrl_ctx *, const mrl_rollout *, const CollectArgs &, int32_t *);
extern template int launch_collect16_t<256, 2>(mrl_ctx *, const mrl_rollout *, const CollectArgs &, int32_t *);

// What mrl_rollout_steps runs a descriptor with.
enum CollectForm {
    FORM_STEPS,      // no fused kernel: the steps are issued one by one
    FORM_WALKER,     // collect_walkers.hpp
    FORM_ROWS16      // collect16.hpp
};
struct CollectPlan {
    CollectForm form;
    int H, act;   // hidden width; 1: ReLU, 2: tanh
};

// Actor and critic must be the agents' nets: two equal hidden layers of 64, 128 or 256 and the env's heads.
static bool agent_nets(const mrl_rollout *r, int obs, int head, bool gauss, int *H, int *act) {
    const mrl_mlp_desc &a = r->actor, &c = r->critic;
    if (a.n_layers != 3 || c.n_layers != 3) return false;
    const int k0 = a.layers[0].kind, h = a.layers[0].out_dim;
    if (k0 != MRL_LINEAR_RELU && k0 != MRL_LINEAR_TANH) return false;
    if (h != 64 && h != 128 && h != 256) return false;
    for (const mrl_mlp_desc *d : {&a, &c}) {
        if (d->layers[0].kind != k0 || d->layers[1].kind != k0) return false;
        if (d->layers[0].in_dim != obs || d->layers[0].out_dim != h || d->layers[1].out_dim != h) return false;
    }
    if (a.layers[2].kind != (gauss ? MRL_STOCHASTIC_ACTOR : MRL_LINEAR) || c.layers[2].kind != MRL_LINEAR) return false;
    if (a.layers[2].out_dim > PA_MAX || (head > 0 && a.layers[2].out_dim != head) || c.layers[2].out_dim != 1) return false;
    *H = h;
    *act = (k0 == MRL_LINEAR_RELU) ? 1 : 2;
    return true;
}

static CollectPlan collect_plan(const mrl_rollout *r, int n_cus) {
    const bool gauss = r->num_actions == 0;
    CollectPlan p{FORM_STEPS, 0, 0};
    const int id = r->env_id;
    int obs = 0, head = 0;
    if (id == MRL_ENV_BIPEDAL) { obs = BipedalWalker::OBS; head = BipedalWalker::ACT_W; }
    else if (id == MRL_ENV_HALFCHEETAH) { obs = HalfCheetah::OBS; head = HalfCheetah::ACT_W; }
    else if (id == MRL_ENV_CARRACING) { obs = cr::OBS; head = cr::ACT; }
    else if (id == MRL_ENV_HOPPER_PLANAR) { obs = planar::Hopper::OBS; head = planar::Hopper::ACT; }
    else if (id == MRL_ENV_WALKER2D_PLANAR) { obs = planar::Walker2d::OBS; head = planar::Walker2d::ACT; }
    if (head > 0) {
        // (the planar rows hold doubles; the weight rows are read with 16-byte loads)
        if (id >= MRL_ENV_HOPPER_PLANAR && reinterpret_cast<uintptr_t>(r->states) % 8 != 0) return p;
        if (reinterpret_cast<uintptr_t>(r->actor_params) % 16 != 0 || reinterpret_cast<uintptr_t>(r->critic_params) % 16 != 0)
            return p;
        if (!gauss || !agent_nets(r, obs, head, true, &p.H, &p.act)) return p;
        // Up to this many envs per CU the walkers' fused kernels are the faster way; with more, their 16-env workgroups
        // come round after round while the stand-alone kernels fill the chip.  us per step, fused against two launches,
        // hidden width 64 / 256:
        //   HalfCheetah (one workgroup per CU)  4096 envs 39 / 44 : 49 / 63,  8192 envs 78 / 88 : 49 / 75;
        //   Walker2d  4096 envs 9.2 / 16.2 : 17.3 / 31.7,  4200 envs 18.3 / 32.1 : 21.8 / 47.7,  8192 envs 18.4 / 32.3 : 19.2 / 44.7
        //     (width 128 22.6 : 27.2),  16384 envs 37 / 64 : 31 / 76 (128 45 : 36);
        //   CarRacing  4096 envs 20 / 31 : 28 / 41,  8192 envs 39 / 61 : 41 / 65,  16384 envs 76 / 121 : 72 / 116;
        //   Hopper  8192 envs 6.9 / 27 : 14.3 / 39,  16384 envs 19.5 / 54 : 25 / 68,  32768 envs 33 / 107 : 35 / 126;
        //   BipedalWalker  4096 envs 26 / 31 : 39 / 53,  8192 envs 51 / 62 : 65 / 91,  12288 envs 77 / 93 : 84 / 127,
        //     16384 envs 102 / 123 : 90 / 133.
        // (The lines were drawn before the fused kernels had their present times: at width 256 Walker2d, Hopper and BipedalWalker,
        // at 64 Walker2d and Hopper are ahead some way beyond theirs.)
        int envs_per_cu = 32;
        if (id == MRL_ENV_HALFCHEETAH || (id == MRL_ENV_WALKER2D_PLANAR && p.H == 64)) envs_per_cu = 16;
        else if (id == MRL_ENV_BIPEDAL && p.H == 256) envs_per_cu = 48;
        else if (id == MRL_ENV_HOPPER_PLANAR) envs_per_cu = 64;
        if (r->n_envs <= envs_per_cu * n_cus) p.form = FORM_WALKER;
        return p;
    }
    if ((id == MRL_ENV_LUNARLANDER && !gauss) || (id == MRL_ENV_LUNARLANDER_CONTINUOUS && gauss)) {
        if (!agent_nets(r, LunarLander::OBS, 0, gauss, &p.H, &p.act)) return p;
        // Hidden width 256: always in one launch.  The narrower nets up to 128 envs per CU, beyond which the stand-alone
        // kernels fill the chip (their env step runs one lane per env).  us per step, one launch : two per step, at
        // 16384 / 32768 / 65536 envs: H = 64 28 : 53, 53 : 68, 103 : 94; H = 128 35 : 59, 68 : 81, 137 : 126; H = 256
        // 59 : 94, 116 : 152, 229 : 268.
        if (p.H == 256 || r->n_envs <= 8 * n_cus * PR16) p.form = FORM_ROWS16;
        return p;
    }
    if (id == MRL_ENV_CARTPOLE && !gauss) obs = cartpole::OBS;
    else if (id == MRL_ENV_PENDULUM && gauss) obs = pendulum::OBS;
    else return p;
    if (!agent_nets(r, obs, 0, gauss, &p.H, &p.act)) return p;
    p.form = FORM_ROWS16;
    return p;
}

}  // namespace mrl

using namespace mrl;

extern "C" {

int mrl_rollout_fused(const mrl_rollout *r) {
    if (r == nullptr) return 0;
    // (the current device, which is the context's where the call is made beside mrl_rollout_steps; without one, an MI355X)
    int device = 0, n_cus = 0;
    if (hipGetDevice(&device) != hipSuccess ||
        hipDeviceGetAttribute(&n_cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) {
        (void)hipGetLastError();
        n_cus = 256;
    }
    return collect_plan(r, n_cus).form != FORM_STEPS ? 1 : 0;
}

int mrl_rollout_steps(mrl_ctx *ctx, const mrl_rollout *r, int t0, int n_steps, uint32_t sample_seed,
                      uint32_t sample_stride, uint64_t step_seed, uint64_t step_stride, uint64_t reset_seed,
                      uint64_t reset_stride) {
    MRL_CHECK_ARG(ctx && r, "mrl_rollout_steps: NULL argument");
    MRL_CHECK_ARG(t0 >= 0 && n_steps >= 0, "mrl_rollout_steps: bad step range");
    if (n_steps == 0) return MRL_OK;
    const bool gauss = r->num_actions == 0;
    const CollectPlan plan = collect_plan(r, ctx->n_cus);
    if (plan.form == FORM_STEPS) {
        for (int k = 0; k < n_steps; ++k) {
            int rc = mrl_rollout_step(ctx, r, t0 + k, sample_seed + (uint32_t)k * sample_stride,
                                      step_seed + (uint64_t)k * step_stride, reset_seed + (uint64_t)k * reset_stride);
            if (rc) return rc;
        }
        return MRL_OK;
    }
    MRL_CHECK_ARG(r->n_envs > 0, "mrl_rollout_steps: bad sizes");
    MRL_CHECK_ARG(r->states && r->obs && r->actor_params && r->critic_params && r->r_obs && r->r_actions &&
                      r->r_log_probs && r->r_values && r->r_rewards && r->r_dones && r->ep_return &&
                      r->ep_length && r->done_returns && r->done_lengths && r->done_count,
                  "mrl_rollout_steps: NULL buffer in descriptor");
    int ss, od, na, ad;
    int rc = mrl_env_dims(r->env_id, &ss, &od, &na, &ad);
    if (rc) return rc;
    MRL_CHECK_ARG(od == r->obs_dim && (gauss ? (ad > 0 && mrl_mlp_out_dim(&r->actor) == 2 * ad)
                                             : (na == r->num_actions && mrl_mlp_out_dim(&r->actor) == na)),
                  "mrl_rollout_steps: descriptor does not match the env's observation / action space");
    const float *shapes = ctx->ll_shapes;
    CollectArgs a{};
    a.states = r->states; a.obs = r->obs;
    a.actor_p = r->actor_params; a.critic_p = r->critic_params; a.shapes = shapes;
    a.n_envs = r->n_envs; a.A = gauss ? ad : na; a.t0 = t0; a.n_steps = n_steps;
    a.sample_seed = sample_seed; a.sample_stride = sample_stride;
    a.reset_seed = reset_seed; a.reset_stride = reset_stride;
    a.r_obs = r->r_obs; a.r_actions = r->r_actions; a.r_logp = r->r_log_probs; a.r_values = r->r_values;
    a.r_rewards = r->r_rewards; a.r_dones = r->r_dones;
    a.acc = Accounting{r->r_rewards, r->r_dones, r->ep_return, r->ep_length, r->done_returns, r->done_lengths,
                       r->done_count, r->done_cap};
    a.spin_limit = ctx->spin_limit;
    a.sync_error = ctx->sync_error;
    a.car_trait_form = ctx->car_trait_form;
    int32_t *side = nullptr;
    if (r->env_id == MRL_ENV_CARTPOLE) {
        rc = cartpole_side(ctx, r->states, r->n_envs, &side);
        if (rc) return rc;
    }
    profile_step_begin(ctx);
    profile_mark(ctx, -1);
    const bool w = plan.form == FORM_WALKER, relu = plan.act == 1;
#define MRL_COLLECT(HH)                                                                                     \
    rc = w ? (relu ? launch_collect_walker_t<HH, 1>(ctx, r, a) : launch_collect_walker_t<HH, 2>(ctx, r, a)) \
           : (relu ? launch_collect16_t<HH, 1>(ctx, r, a, side) : launch_collect16_t<HH, 2>(ctx, r, a, side))
    if (plan.H == 64) MRL_COLLECT(64);
    else if (plan.H == 128) MRL_COLLECT(128);
    else MRL_COLLECT(256);
#undef MRL_COLLECT
    if (rc) return rc;
    MRL_CHECK_LAUNCH();
    profile_mark(ctx, MRL_PHASE_COLLECT);
    profile_step_end(ctx);
    return MRL_OK;
}

}  // extern "C"
