"""GPU: gradients and optimiser state of the minibatch update may lie on any float (slices of one vector for all nets): the
same update bit for bit as on buffers of their own, and nothing written beside them; also where the action is wider than the
observation, which the layer-by-layer update refuses."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H", [64, 128, 256])
@pytest.mark.parametrize("IN,A,cont", [(8, 4, False), (3, 6, True)])
def test_gradients_and_state_on_any_float(mrl, H, IN, A, cont):
    ctx = mrl.DeviceContext("cuda:0")
    E = type("E", (), dict(ENV_ID=-1, STATE_SIZE=IN, OBS_DIM=IN, NUM_ACTIONS=0 if cont else A, ACTION_DIM=A if cont else 0))
    lay = mrl.LinearTanh if cont else mrl.LinearReLU
    actor = mrl.seq(lay(IN, H), lay(H, H), mrl.StochasticActor(H, A) if cont else mrl.Linear(H, A))
    critic = mrl.seq(lay(IN, H), lay(H, H), mrl.Linear(H, 1))
    MB, n_mb = 45, 3
    g = torch.Generator(device="cuda").manual_seed(H)
    rnd = lambda n, s: (torch.rand(n, device="cuda", generator=g) - 0.5) * 2 * s
    params = rnd(actor.PARAM_SIZE, 0.1), rnd(critic.PARAM_SIZE, 0.1)
    total = MB * n_mb
    rows = rnd(total * IN, 1), rnd(total, 0.05) - 1.4, rnd(total, 1), rnd(total, 1), rnd(total, 1)
    acts = rnd(total * A, 1) if cont else torch.randint(0, A, (total,), device="cuda", generator=g).float()
    perm = torch.randperm(total, device="cuda", generator=g).to(torch.int32)

    def run(off):
        rb = mrl.ppo.RolloutBuffers(ctx, E, actor, critic, MB, n_mb)
        rb.actor_params, rb.critic_params = params[0].clone(), params[1].clone()
        for dst, src in ((rb.r_obs, rows[0]), (rb.r_log_probs, rows[1]), (rb.r_values, rows[2]), (rb.r_actions, acts)):
            dst.copy_(src)
        cls = mrl.ppo.ContinuousUpdate if cont else mrl.ppo.DiscreteUpdate
        upd = cls(ctx, rb, MB, mrl.Adam(lr=1e-2), mrl.Adam(lr=1e-2), target_kl=1e9)
        upd.advantages.copy_(rows[3])
        upd.returns.copy_(rows[4])
        names = ("actor_grads", "critic_grads", "actor_state", "critic_state")
        guards = []
        if off:
            sizes = [getattr(upd, n).numel() for n in names]
            flat, at = torch.full((sum(sizes) + 4 * (off + 3),), 7.0, device="cuda"), 0
            for n, size in zip(names, sizes):
                lead = (at + off) if (at + off) % 4 else at + off + 1      # never on 16 bytes
                guards += [flat[at:lead]]
                part = flat[lead:lead + size]
                assert part.data_ptr() % 16 != 0
                part.zero_()
                setattr(upd, n, part)
                at = lead + size
            guards.append(flat[at:])
        upd.reset_kl()
        upd.run_epoch(perm)
        ctx.synchronize()
        assert all(bool((t == 7.0).all()) for t in guards)
        return [rb.actor_params, rb.critic_params] + [getattr(upd, n).clone() for n in names]

    want = run(0)
    assert float(want[2].abs().max()) > 0
    for off in (1, 2, 3):
        for a, b in zip(want, run(off)):
            assert torch.equal(a, b)
