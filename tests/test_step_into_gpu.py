"""Env.step_into against Env.step with its out columns copied: observations, out, hash, state and
the reward and done rows, in both builds of the step; and workgroups of several worlds against the
same worlds stepped one a workgroup."""
import importlib
import pathlib
import re

import pytest
import torch

pytestmark = pytest.mark.gpu


def seam_sizes():
    """(worlds, monsters, rng_mode) in both builds with two workgroups of several worlds before the
    one-world tail and every remainder between them, from the split the kernels are built with."""
    source = pathlib.Path(__file__).resolve().parents[1] / 'dcss-auto_amd' / 'csrc' / 'd1_env.hip'
    k = {name: int(v) for name, v in re.findall(r'\b((?:STEP|CROWD)_(?:TAIL|WPB)) = (\d+)', source.read_text())}
    assert k['STEP_WPB'] > 1 and k['CROWD_WPB'] > 1
    sizes = []
    for build, monsters in (('STEP', (8, 3)), ('CROWD', (40, 12))):
        for rest in range(k[f'{build}_WPB']):
            for rng_mode in (0, 1):
                sizes.append((k[f'{build}_TAIL'] + 2 * k[f'{build}_WPB'] + rest, monsters[rest % 2], rng_mode))
    return sizes


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


@pytest.mark.parametrize('worlds,monsters,rng_mode', seam_sizes())
def test_worlds_of_one_workgroup_step_as_alone(pkg, worlds, monsters, rng_mode):
    """A whole-batch step has workgroups of several worlds and then one-world ones; slices shorter
    than that tail have one-world workgroups only. Every world's rows are the same, with every action
    and episodes that end and reset within a workgroup."""
    print(f'[seam] {worlds} worlds, {monsters} monsters, rng {rng_mode}', flush=True)
    cfg = pkg.make_config(monsters, rng_mode=rng_mode, awake_pct=50, limit=6)
    whole, into, alone = (pkg.Env(worlds, cfg, seed=3) for _ in range(3))
    g = torch.Generator(device='cuda').manual_seed(2)
    obs = torch.empty(worlds * 1800, dtype=torch.uint8, device='cuda')
    reward = torch.empty(worlds, device='cuda')
    done = torch.empty(worlds, dtype=torch.uint8, device='cuda')
    cuts = [0, 3, worlds // 3, 2 * worlds // 3, worlds]
    ended = torch.zeros(worlds, device='cuda')
    for _ in range(9):
        act = torch.randint(0, 19, (worlds,), generator=g, device='cuda', dtype=torch.int64)
        whole.step(act)
        into.step_into(act, obs, reward, done)
        for lo, hi in zip(cuts, cuts[1:]):
            alone.step_rows(lo, hi, act)
        for env, seen in ((whole, whole.obs), (into, obs)):
            assert torch.equal(env.state, alone.state) and torch.equal(env.out, alone.out)
            assert torch.equal(seen.view_as(alone.obs), alone.obs)
        assert torch.equal(whole.hash, into.hash)
        assert torch.equal(reward, alone.out[:, 0]) and torch.equal(done, alone.out[:, 1].to(torch.uint8))
        ended += alone.out[:, 1]
    assert bool((ended[:6] > 0).all())   # also in the first workgroups


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
