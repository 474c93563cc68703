"""Timed cases: the calls that a user of this package makes, each over the range of sizes it is made with.

Kinds of work, all through the package's public entry points:

  act      ppo.policy_step for environments that live on the host (the loop of train_gpu_cpu_env): actor and critic
           forward, sampling and the rollout stores for a handful to a few thousand observations;
  env      one step_autoreset_kernel_gpu of an environment class, as a caller with a policy of its own makes it;
  rollout  ppo.rollout_steps: the collection loop of train_gpu, policy and environment on the device;
  update   PPOUpdate.update on a collected rollout: bootstrap values, GAE, advantage normalisation, and epochs of
           shuffled minibatches with the KL test armed, as train_gpu runs it;
  train    an agent's train_gpu for one rollout: buffers, reset, rollout, update and the episode read-back;
  mlp      Network.forward_gpu / backward_gpu / update_gpu, the layer API under a loss of the caller's;
  gae      compute_gae and normalize_advantages on a rollout's buffers.

Everything is float32 (the planar environments keep Float64 state), on the device, made from the seed.
"""
import importlib
import math

import torch

mrl = importlib.import_module("mojo-rl_amd")
ppo = mrl.ppo

# name -> (class, bytes of live state, action, observation, reward and done that a step reads or writes once)
ENVS = {
    "cartpole": (mrl.CartPoleEnv, 60),
    "pendulum": (mrl.PendulumV2, 72),
    "lunarlander": (mrl.LunarLanderV2, 672),
    "lunarlander_continuous": (mrl.LunarLanderV2Continuous, 676),
    "bipedal": (mrl.BipedalWalkerV2, 3964),
    "halfcheetah": (mrl.HalfCheetahPlanarV2, 1112),
    "carracing": (mrl.CarRacingV2, 11120),
    "hopper": (mrl.HopperPlanar, 560),
    "walker2d": (mrl.Walker2dPlanar, 884),
}
PLANAR = ("hopper", "walker2d")     # rows hold Float64 values as pairs of floats
PREROLL = 128                       # steps that take freshly reset envs to their usual mix of flight, contacts and resets


def listed():
    return [
        # sixteen host environments asking for their next actions: the smallest call, all latency
        dict(name="act_cartpole_16", kind="act", env="cartpole", n=16, hidden=64),
        # a caller's own loop over a ragged thousand envs of the rigid-body engine
        dict(name="env_lunarlander_1000", kind="env", env="lunarlander", n=1000),
        # data generation at a batch that fills the chip many times over
        dict(name="env_bipedal_65536", kind="env", env="bipedal", n=65536),
        # the agents' default sizes (1024 envs, 128 steps, hidden width 64)
        dict(name="rollout_cartpole_1024", kind="rollout", env="cartpole", n=1024, steps=128, hidden=64),
        # the benchmark's default workload
        dict(name="rollout_lunarlander_8192", kind="rollout", env="lunarlander", n=8192, steps=64, hidden=256),
        # a continuous-control benchmark workload
        dict(name="rollout_halfcheetah_4096", kind="rollout", env="halfcheetah", n=4096, steps=32, hidden=256),
        # the default hidden width on a rigid-body env, a ragged number of envs
        dict(name="rollout_lunarlander_777_h64", kind="rollout", env="lunarlander", n=777, steps=128, hidden=64),
        # train_gpu with every default of DeepPPOAgent: 512 minibatches of 256 per epoch, up to four epochs (the KL stop
        # ends a first update after the first)
        dict(name="train_cartpole_default", kind="train", env="cartpole", n=1024, steps=128, hidden=64, minibatch=256,
             epochs=4, clip_value=True, critic_lr=1e-3),
        # the update of a continuous-control run at the benchmark's sizes
        dict(name="update_halfcheetah_4096", kind="update", env="halfcheetah", n=4096, steps=32, hidden=256,
             minibatch=4096, epochs=2, clip_value=False, critic_lr=3e-4),
        # a width between the two that the configurations name, an uneven minibatch
        dict(name="update_walker2d_h128", kind="update", env="walker2d", n=500, steps=64, hidden=128, minibatch=1000,
             epochs=2, clip_value=False, critic_lr=3e-4),
        # one gradient step of a 256-wide tanh network on a loss of the caller's
        dict(name="mlp_24_256_256_8", kind="mlp", batch=4096, inputs=24, hidden=256, outputs=8, tanh=True, grad_in=True),
        # advantages of a thousand-step rollout of 4096 envs
        dict(name="gae_1000x4096", kind="gae", steps=1000, n=4096),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["act", "env", "rollout", "rollout", "update", "update", "train", "mlp", "gae"])
    env = rng.choice(sorted(ENVS))
    hidden = rng.choice([64, 128, 256])
    if kind == "act":
        return dict(kind=kind, env=env, n=_log_int(rng, 1, 4096), hidden=hidden)
    if kind == "env":
        return dict(kind=kind, env=env, n=_log_int(rng, 64, 65536 if env in ("bipedal", "halfcheetah", "carracing") else 262144))
    if kind == "gae":
        return dict(kind=kind, steps=_log_int(rng, 32, 1000), n=_log_int(rng, 64, 4096))
    if kind == "mlp":
        return dict(kind=kind, batch=_log_int(rng, 32, 16384), inputs=rng.randint(3, 32), hidden=hidden,
                    outputs=rng.randint(1, 8), tanh=rng.random() < 0.5, grad_in=rng.random() < 0.5)
    n, steps = _log_int(rng, 64, 8192), _log_int(rng, 16, 128)
    if kind == "rollout":
        return dict(kind=kind, env=env, n=n, steps=steps, hidden=hidden)
    n, steps = _log_int(rng, 64, 4096), _log_int(rng, 16, 64)
    minibatch = min(_log_int(rng, 64, 8192), n * steps)
    # at most 48 minibatches: a sample next to a clip boundary that falls on its other side changes every later step
    n = min(n, 3 * minibatch)
    steps = min(steps, 48 * minibatch // n)
    epochs = rng.choice([1, 2]) if kind == "update" and 2 * n * steps <= 48 * minibatch else 1
    return dict(kind=kind, env=env, n=n, steps=steps, hidden=hidden, minibatch=minibatch, epochs=epochs, clip_value=False,
                critic_lr=3e-4)


class _State:
    pass


def _nets(env, hidden):
    """Actor and critic as the agents build them: ReLU layers and logits, or tanh layers and a Gaussian head."""
    E = ENVS[env][0]
    lay = mrl.LinearReLU if E.NUM_ACTIONS else mrl.LinearTanh
    head = mrl.Linear(hidden, E.NUM_ACTIONS) if E.NUM_ACTIONS else mrl.StochasticActor(hidden, E.ACTION_DIM)
    return (mrl.seq(lay(E.OBS_DIM, hidden), lay(hidden, hidden), head),
            mrl.seq(lay(E.OBS_DIM, hidden), lay(hidden, hidden), mrl.Linear(hidden, 1)))


def _buffers(s, case, seed, steps):
    """Rollout buffers with networks initialised as the agents initialise theirs and freshly reset envs."""
    E, n, H = ENVS[case["env"]][0], case["n"], case["hidden"]
    actor, critic = _nets(case["env"], H)
    init = mrl.Xavier if E.NUM_ACTIONS else mrl.Kaiming
    s.anet = mrl.Network(s.ctx, actor, mrl.Adam(lr=3e-4), init(seed=2 * seed + 1))
    s.cnet = mrl.Network(s.ctx, critic, mrl.Adam(lr=case.get("critic_lr", 1e-3)), init(seed=2 * seed + 2))
    if not E.NUM_ACTIONS:
        mrl.init_params_small(s.ctx, s.anet.params, E.OBS_DIM * H + H + H * H + H, H, E.ACTION_DIM, seed=2 * seed + 3)
    s.rb = rb = ppo.RolloutBuffers(s.ctx, E, actor, critic, n, steps, done_cap=max(1024, n * max(steps, PREROLL)))
    rb.actor_params, rb.critic_params = s.anet.params, s.cnet.params
    if case["env"] == "cartpole":
        s.counters = torch.zeros(n, dtype=torch.int32, device=s.ctx.device)
        E.bind_step_counters(s.ctx, rb.states, s.counters)
    E.reset_kernel_gpu(s.ctx, rb.states, seed)
    rb.obs.copy_(rb.states.view(n, E.STATE_SIZE)[:, :E.OBS_DIM].reshape(-1))
    s.desc = rb.descriptor()
    s.taken = seed * 1000003 % 2**31


def _collect(s, steps):
    """One rollout with train_gpu's seeds."""
    n, ts = s.rb.n_envs, s.taken
    ppo.rollout_steps(s.ctx, s.desc, 0, steps, ts * 2654435761, n * 2654435761 + 7919,
                      ts * 1103515245, n * 1103515245 + 12345, ts * 1013904223, n * 1013904223 + 2654435761)
    s.taken += n * steps


def _states(case, states):
    return states.view(torch.int32) if case["env"] in PLANAR else states


def prepare(case, seed):
    kind = case["kind"]
    s = _State()
    s.case, s.ctx, s.k = case, mrl.DeviceContext("cuda:0"), 0
    dev = s.ctx.device
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    if kind == "act":
        s.steps = 32
        _buffers(s, case, seed, s.steps)
        s.rb.obs.normal_(generator=g)
        s.actions = torch.zeros(case["n"] * s.rb.act_width, device=dev)
    elif kind == "env":
        E, n = ENVS[case["env"]][0], case["n"]
        s.states = torch.zeros(n * E.STATE_SIZE, device=dev)
        if case["env"] == "cartpole":
            s.counters = torch.zeros(n, dtype=torch.int32, device=dev)
            E.bind_step_counters(s.ctx, s.states, s.counters)
        E.reset_kernel_gpu(s.ctx, s.states, seed)
        s.rewards, s.dones, s.obs = (torch.zeros(n * w, device=dev) for w in (1, 1, E.OBS_DIM))
        # eight sets of random actions, taken in turn
        if E.NUM_ACTIONS:
            s.actions = torch.randint(0, E.NUM_ACTIONS, (8, n), device=dev, generator=g).float()
        else:
            s.actions = torch.rand(8, n * E.ACTION_DIM, device=dev, generator=g) * 2 - 1
        for _ in range(PREROLL):
            run(s)
    elif kind == "rollout":
        _buffers(s, case, seed, case["steps"])
        for _ in range(-(-PREROLL // case["steps"])):
            _collect(s, case["steps"])
    elif kind == "update":
        _buffers(s, case, seed, case["steps"])
        _collect(s, case["steps"])
        cls = ppo.ContinuousUpdate if s.rb.continuous else ppo.DiscreteUpdate
        s.upd = cls(s.ctx, s.rb, case["minibatch"], s.anet.optimizer, s.cnet.optimizer, clip_value=case["clip_value"],
                    target_kl=0.02 if s.rb.continuous else 0.015)
        s.start = (s.anet.params.clone(), s.cnet.params.clone())
    elif kind == "train":
        E = ENVS[case["env"]][0]
        cls, out = (mrl.DeepPPOAgent, E.NUM_ACTIONS) if E.NUM_ACTIONS else (mrl.DeepPPOContinuousAgent, E.ACTION_DIM)
        s.agent = cls(E.OBS_DIM, out, hidden_dim=case["hidden"], rollout_len=case["steps"], n_envs=case["n"],
                      gpu_minibatch_size=case["minibatch"], num_epochs=case["epochs"], clip_value=case["clip_value"],
                      critic_lr=case["critic_lr"], init_seed=seed)
        s.agent.build_networks(s.ctx)
        s.seed = seed
        s.start = (s.agent.actor.params.clone(), s.agent.critic.params.clone())
    elif kind == "mlp":
        lay = mrl.LinearTanh if case["tanh"] else mrl.LinearReLU
        b, i, h, o = case["batch"], case["inputs"], case["hidden"], case["outputs"]
        model = mrl.seq(lay(i, h), lay(h, h), mrl.Linear(h, o))
        s.net = mrl.Network(s.ctx, model, mrl.Adam(lr=3e-4), mrl.Kaiming(seed=seed))
        s.x = torch.randn(b * i, device=dev, generator=g)
        s.target = torch.randn(b * o, device=dev, generator=g)
        s.out, s.cache = torch.empty(b * o, device=dev), torch.empty(b * model.CACHE_SIZE, device=dev)
        s.grad_in = torch.empty(b * i, device=dev) if case["grad_in"] else None
    elif kind == "gae":
        t, n = case["steps"], case["n"]
        s.rewards, s.values = (torch.randn(t * n, device=dev, generator=g) for _ in range(2))
        s.dones = (torch.rand(t * n, device=dev, generator=g) < 0.01).float()      # episodes of about a hundred steps
        s.bootstrap = torch.randn(n, device=dev, generator=g)
        s.adv, s.ret = torch.empty(t * n, device=dev), torch.empty(t * n, device=dev)
    else:
        raise ValueError("unknown kind %r" % kind)
    return s


def run(s):
    case, kind, k = s.case, s.case["kind"], s.k
    s.k += 1
    if kind == "act":
        rb, n, t = s.rb, case["n"], k % s.steps
        ppo.policy_step(s.ctx, rb, t, 7919 * k, s.actions)
        row = slice(t * n, (t + 1) * n)
        od, aw = rb.env.OBS_DIM, rb.act_width
        return {"actions": s.actions, "r_obs": rb.r_obs[t * n * od:(t + 1) * n * od],
                "r_actions": rb.r_actions[t * n * aw:(t + 1) * n * aw], "log_probs": rb.r_log_probs[row], "values": rb.r_values[row]}
    if kind == "env":
        E = ENVS[case["env"]][0]
        E.step_autoreset_kernel_gpu(s.ctx, s.states, s.actions[k % 8], s.rewards, s.dones, s.obs, k, 100003 + k)
        return {"states": _states(case, s.states), "rewards": s.rewards, "dones": s.dones, "obs": s.obs}
    if kind == "rollout":
        rb = s.rb
        rb.done_count.zero_()
        _collect(s, case["steps"])
        return {"states": _states(case, rb.states), "obs": rb.obs, "r_obs": rb.r_obs, "r_actions": rb.r_actions,
                "log_probs": rb.r_log_probs, "values": rb.r_values, "rewards": rb.r_rewards, "dones": rb.r_dones,
                "ep_return": rb.ep_return, "ep_length": rb.ep_length, "done_count": rb.done_count}
    if kind == "update":
        # the update phase of a training iteration starts from the weights that collected the rollout
        _restart(s.anet, s.start[0])
        _restart(s.cnet, s.start[1])
        upd = s.upd
        upd.actor_state.zero_()
        upd.critic_state.zero_()
        upd.update(case["epochs"], seed=k)
        return {"actor": s.anet.params, "critic": s.cnet.params, "actor_state": upd.actor_state, "critic_state": upd.critic_state,
                "actor_grads": upd.actor_grads, "critic_grads": upd.critic_grads, "advantages": upd.advantages, "returns": upd.returns}
    if kind == "train":
        a = s.agent
        for net, start in ((a.actor, s.start[0]), (a.critic, s.start[1])):
            _restart(net, start)
            net.optimizer_state.zero_()
        a.train_gpu(s.ctx, ENVS[case["env"]][0], num_episodes=1 << 30, max_rollouts=1, seed=s.seed + k)
        rb, upd = a.rb, a.upd
        return {"actor": a.actor.params, "critic": a.critic.params, "actor_state": a.actor.optimizer_state,
                "critic_state": a.critic.optimizer_state, "advantages": upd.advantages, "returns": upd.returns, "obs": rb.obs,
                "r_obs": rb.r_obs, "r_actions": rb.r_actions, "log_probs": rb.r_log_probs, "values": rb.r_values,
                "rewards": rb.r_rewards, "dones": rb.r_dones}
    if kind == "mlp":
        s.net.forward_gpu(s.out, s.x, s.cache)
        grad = (s.out - s.target) * (2.0 / s.out.numel())       # mean squared error
        s.net.backward_gpu(s.grad_in, grad, s.cache)
        s.net.update_gpu()
        return {"out": s.out, "grads": s.net.grads, "params": s.net.params, "optimizer_state": s.net.optimizer_state,
                "grad_in": s.grad_in}
    ppo.compute_gae(s.ctx, s.rewards, s.values, s.dones, s.bootstrap, 0.99, 0.95, s.adv, s.ret)
    ppo.normalize_advantages(s.ctx, s.adv)
    return {"advantages": s.adv, "returns": s.ret}


def _restart(net, params):
    net.params.copy_(params)
    net.optimizer.t = 0


def _dims(case):
    """(forward flops per row of actor + critic, floats of a rollout row, parameters of the two nets)."""
    E, H = ENVS[case["env"]][0], case["hidden"]
    a = E.NUM_ACTIONS or E.ACTION_DIM
    flops = 2 * (2 * (E.OBS_DIM * H + H * H) + H * (a + 1))
    params = 2 * ((E.OBS_DIM + 1) * H + (H + 1) * H) + (H + 1) * (a + 1)
    return flops, E.OBS_DIM + (E.ACTION_DIM or 1) + 2, params


def _work_rollout(case, steps):
    flops, row, params = _dims(case)
    return {"flops": case["n"] * steps * flops,
            "bytes": 4 * (case["n"] * steps * (row + 2) + params) + ENVS[case["env"]][1] * case["n"]}


def _work_update(case, epochs):
    flops, row, params = _dims(case)
    total = case["n"] * case["steps"]
    minibatches = total // case["minibatch"] * epochs
    # forward, input gradient and weight gradient of every sample; each sample's row, advantage and return once per
    # epoch; parameters, gradients and Adam's two moments once per minibatch; GAE's five arrays
    return {"flops": 3 * minibatches * case["minibatch"] * flops,
            "bytes": 4 * (minibatches * case["minibatch"] * (row + 3) + minibatches * 7 * params + 5 * total)}


def work(case):
    kind = case["kind"]
    if kind == "act":
        flops, row, params = _dims(case)
        return {"flops": case["n"] * flops, "bytes": 4 * (case["n"] * 2 * row + params)}
    if kind == "env":
        return {"flops": 0, "bytes": case["n"] * ENVS[case["env"]][1]}
    if kind == "rollout":
        return _work_rollout(case, case["steps"])
    if kind == "update":
        return _work_update(case, case["epochs"])
    if kind == "train":
        r, u = _work_rollout(case, case["steps"]), _work_update(case, 1)
        return {m: r[m] + u[m] for m in r}
    if kind == "mlp":
        b, i, h, o = case["batch"], case["inputs"], case["hidden"], case["outputs"]
        params = (i + 1) * h + (h + 1) * h + (h + 1) * o
        return {"flops": 6 * b * (i * h + h * h + h * o), "bytes": 4 * (b * (2 * i + 3 * o) + 7 * params)}
    return {"flops": 10 * case["steps"] * case["n"], "bytes": 4 * case["n"] * (7 * case["steps"] + 1)}


def tolerance(case):
    # Four times and more what the same pass shows with its sums in another order (the rows of every minibatch shuffled)
    # or in Float64.  Forward passes: 3e-7, single values 2e-6.  Updates: 5e-7 (single values 3e-5) as a rule, up to a
    # few 1e-4 (single values 1e-2) where a sample sits next to a clip boundary or a critic's gradients nearly cancel.
    if case["kind"] == "env":
        return "exact"
    if case["kind"] in ("update", "train"):
        return {"rel": 1e-3, "max": 0.05}
    if case["kind"] == "mlp":
        return {"rel": 5e-6, "max": 1e-3}
    return {"rel": 2e-6, "max": 5e-5}
