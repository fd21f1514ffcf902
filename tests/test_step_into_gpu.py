"""Env.step_into against Env.step with its out columns copied: observations, out, hash, state and
the reward and done rows, in both builds of the step and around the workgroups' world counts."""
import importlib

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('worlds,monsters', [(1, 8), (5, 8), (4097, 8), (4103, 3), (3, 40), (8195, 12)])
def test_step_into_equals_step(pkg, worlds, monsters):
    print(f'[step_into] {worlds} worlds, {monsters} monsters', flush=True)
    cfg = pkg.make_config(monsters, awake_pct=50, limit=6)     # episodes end within the run
    a, b = (pkg.Env(worlds, cfg, seed=3) for _ in range(2))
    g = torch.Generator(device='cuda').manual_seed(1)
    obs = torch.empty(worlds * 1800, dtype=torch.uint8, device='cuda')
    reward = torch.full((worlds + 8,), 9.0, device='cuda')
    done = torch.full((worlds + 8,), 9, dtype=torch.uint8, device='cuda')
    ended = 0
    for _ in range(8):
        act = torch.randint(0, 19, (worlds,), generator=g, device='cuda', dtype=torch.int64)
        want, out = a.step(act)
        b.step_into(act, obs, reward[:worlds], done[:worlds])
        assert torch.equal(obs.view_as(want), want) and torch.equal(b.out, out)
        assert torch.equal(a.hash, b.hash) and torch.equal(a.state, b.state)
        assert torch.equal(reward[:worlds], out[:, 0]) and torch.equal(done[:worlds], out[:, 1].to(torch.uint8))
        ended += int(done[:worlds].sum())
    assert ended > 0 and bool((reward[worlds:] == 9).all()) and bool((done[worlds:] == 9).all())
    with pytest.raises(ValueError):
        b.step_into(act, obs, reward, done[:worlds])


def test_trainer_keeps_an_overridden_step(pkg):
    """An environment with a step of its own is stepped through it."""
    train = importlib.import_module('dcss-auto_amd.train')
    P = importlib.import_module('dcss-auto_amd.policy')

    class Counting(pkg.Env):
        calls = 0

        def step(self, actions, active=None, obs=None):
            self.calls += 1
            return super().step(actions, active=active, obs=obs)

    bufs = []
    for cls in (pkg.Env, Counting):
        env = cls(128, pkg.baseline_config(8), seed=2, hash=False)
        tr = train.Trainer(env, P.Policy(seed=1).cuda(), horizon=8, minibatch=1024, graph=False)
        bufs.append(tr.rollout())
    assert env.calls == 8
    for k in ('obs', 'actions', 'logp', 'values', 'rewards', 'dones', 'bootstrap'):
        assert torch.equal(getattr(bufs[0], k), getattr(bufs[1], k)), k
