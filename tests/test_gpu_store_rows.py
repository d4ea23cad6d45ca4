"""The rollout storage's writes (ppo_store_rows) and act()'s one-launch distribution against the general path: torch
copies, and update / sample / log_prob one after another.  Every written value is the same, bit for bit."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture
def cuda():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    return torch.device("cuda:0")


@pytest.mark.parametrize("n", [1, 3, 1023, 1024, 4097])
def test_row_stores(cuda, n):
    from tt_rsl_rl_amd import ops

    g = torch.Generator("cuda").manual_seed(n)
    rnd = lambda *s: torch.randn(*s, generator=g, device=cuda)  # noqa: E731
    flags = rnd(n, 1) > 0
    rec = rnd(n, 96)
    pairs = [  # destination, source: flat (16-byte pieces or not), records with padding, views off 16 bytes, flags
        (rnd(n, 96), rnd(n, 96)), (rnd(n, 7), rnd(n, 7)), (rec[:, :29], rnd(n, 29)), (rec[:, 32:61], rnd(n, 61)[:, 32:]),
        (rnd(n, 5), rnd(n, 12)[:, 3:8]), (rnd(n * 8 + 1)[1:].view(n, 8), rnd(n, 8)), (rnd(2, n, 16), rnd(2, n, 16)),
        (rnd(n, 29), rnd(1, 29).expand(n, 29)), (rnd(n, 6), rnd(6, n).t()), (rnd(n, 4), rnd(n, 4).double()),
        (rnd(n, 4), rnd(n, 4).cpu()), (rnd(n, 4), rnd(n, 1)), (rnd(0, 4), rnd(0, 4)), (rnd(n, 3), rnd(n, 3).requires_grad_()),
    ] + [(torch.full((n, 1), 9, dtype=torch.uint8, device=cuda), flags.to(t)) for t in
         (torch.float32, torch.bool, torch.uint8, torch.int64, torch.int32)]
    pairs.append((torch.zeros(n, 1, dtype=torch.uint8, device=cuda), 300.0 * rnd(n, 1).abs()))
    rest = rec.clone()
    w = ops.RowStores(cuda)
    with torch.no_grad():
        for d, s in pairs:
            w.copy(d, s)
        w.flush()
    for i, (d, s) in enumerate(pairs):
        want = torch.empty_like(d, memory_format=torch.contiguous_format)
        with torch.no_grad():
            want.copy_(s)
        assert torch.equal(d, want), i
    assert torch.equal(rec[:, 29:32], rest[:, 29:32]) and torch.equal(rec[:, 61:], rest[:, 61:])
    for t in (torch.float32, torch.bool, torch.uint8, torch.int64):
        out, r, v = rnd(n, 1), rnd(n), rnd(n, 1)
        v[0] = float("nan")
        w.bootstrap(out, r, 0.99, v, flags[:, 0].to(t))
        w.flush()
        want = r.clone()
        want += 0.99 * torch.squeeze(v * flags[:, 0].to(t).unsqueeze(1), 1)
        assert torch.equal(out[:, 0].nan_to_num(7.0), want.nan_to_num(7.0)), t


@pytest.mark.parametrize("envs, actions, rnn", [(1, 1, ""), (31, 64, ""), (33, 29, ""), (4097, 13, ""), (65, 12, "lstm")])
def test_act_and_step_match_the_general_path(cuda, envs, actions, rnn):
    """A forward hook on the actor takes act() to the separate calls, rewards of shape [N, 1] the step to torch's."""
    from types import SimpleNamespace

    from tt_rsl_rl_amd.ppo import PPO

    def collect(general):
        torch.manual_seed(0)
        model = dict(class_name="RNNModel" if rnn else "MLPModel", hidden_dims=[32, 32], activation="elu")
        if rnn:
            model.update(rnn_type=rnn, rnn_hidden_dim=64, rnn_num_layers=1)
        cfg = dict(algorithm=dict(class_name="tt_rsl_rl_amd.ppo:PPO"),
                   actor=dict(model, distribution_cfg=dict(class_name="GaussianDistribution", init_std=0.7, std_type="log")),
                   critic=model, obs_groups={"actor": ["policy"], "critic": ["policy"]}, num_steps_per_env=3)
        alg = PPO.construct_algorithm({"policy": torch.zeros(envs, 20)}, SimpleNamespace(num_envs=envs, num_actions=actions),
                                      cfg, "cuda:0")
        alg.train_mode()
        if general:
            alg.actor.register_forward_hook(lambda *a: None)
        assert alg.actor.acts_plainly() is not general
        g = torch.Generator("cuda").manual_seed(5)
        shown = []
        with torch.inference_mode():
            for _ in range(3):
                obs = {"policy": torch.randn(envs, 20, generator=g, device=cuda)}
                rewards, u = torch.randn(envs, generator=g, device=cuda), torch.rand(envs, generator=g, device=cuda)
                kept = rewards.clone()
                a = alg.act(obs)
                shown += [a.clone(), alg.transition.actions_log_prob.clone(), alg.actor.output_std.clone()]
                time_outs = (u < 0.2) if not general else (u < 0.2).cpu()
                alg.process_env_step(obs, rewards, (u < 0.4).long(), {"time_outs": time_outs})
                assert torch.equal(rewards, kept)
        st = alg.storage
        return shown + [st.observations["policy"], st.actions, st.rewards, st.dones, st.values, st.actions_log_prob,
                        *st.distribution_params, *(st.saved_hidden_state_a or ()), *(st.saved_hidden_state_c or ())]

    for i, (x, y) in enumerate(zip(collect(False), collect(True), strict=True)):
        assert torch.equal(x, y), i


def test_sources_made_for_the_call(cuda):
    """Observations that a mapping computes on access are freed with the call that took them: each destination still gets
    its own."""
    from tt_rsl_rl_amd import ops

    src = [torch.full((512, 8), float(i), device=cuda) for i in range(6)]
    dst = [torch.empty(512, 8, device=cuda) for _ in src]
    w = ops.RowStores(cuda)
    for d, s in zip(dst, src):
        w.copy(d, s.clone())
    w.bootstrap(dst[0][:, :1].clone(), src[0][:, 0].clone(), 0.5, src[1][:, :1].clone(), src[2][:, 0].clone())
    w.flush()
    assert all(torch.equal(d, s) for d, s in zip(dst, src)) and not w.items and not w.held
