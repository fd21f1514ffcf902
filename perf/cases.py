"""The work that a user of this framework has it do, as measurable cases.

Every case is one pass through the public Python surface on one GPU: an environment step, the
learning task's decision, a policy forward with its sample, a rollout, GAE, a PPO update. Sizes
are those of BASELINE's configurations (C1 1,024 worlds, C3 65,536 worlds, C4 minibatches of
8,192, C5 262,144 crowded worlds), of the learning task's bench and of smaller runs of the same
loops; `draw` spreads them, ragged ones among them, over the ranges in between.
"""
import importlib
import math

import torch

pkg = importlib.import_module('dcss-auto_amd')
learn = importlib.import_module('dcss-auto_amd.learn')
policy = importlib.import_module('dcss-auto_amd.policy')
ppo = importlib.import_module('dcss-auto_amd.ppo')
train = importlib.import_module('dcss-auto_amd.train')

DEV = 'cuda:0'
RING = 16                  # action rows an environment case walks through, one a pass
# multiply-adds of one sample: the trunk with its 17-row head; the verb and value rows, the
# target MLP's trunk part and one verb's 25 targets of the autoregressive head
TRUNK_FLOPS = 2 * (1800 * 256 + 256 * 256 + 256 * 17)
AR_FLOPS = 2 * (1800 * 256 + 256 * 256 + 256 * 9 + 256 * 64 + 64 * 25)
# forward and backward of one sample without the input gradient of the first layer
PPO_FLOPS = TRUNK_FLOPS + 2 * (1800 * 256 + 2 * 256 * 256 + 2 * 256 * 17)
POLICY_PARAMS = 1800 * 256 + 256 + 256 * 256 + 256 + 256 * 17 + 17
LEARN_BYTES = 7388         # one learning-task decision (observation, mask, outcome, row, memory, floor)


def listed():
    return [
        # C1: the smallest batch that is run in earnest (a debugging or parity run), hashed
        dict(name='env_c1', kind='env', worlds=1024, monsters=8, rules='baseline', hash=True),
        # C3: the rollout's environment step, no hash
        dict(name='env_c3', kind='env', worlds=65536, monsters=8, rules='baseline', hash=False),
        # the reference's 24-enemy task on map 1057 with its own RNG, a ragged batch
        dict(name='env_ref24', kind='env', worlds=4133, monsters=24, rules='reference', hash=True),
        # C5: 40 monsters, half of them awake
        dict(name='env_c5', kind='env', worlds=262144, monsters=40, rules='stress', hash=False),
        # the learning task's drop-in loop: controller, then step, at its bench size
        dict(name='learn_64k', kind='learn', worlds=65536, maps=1, clump=0),
        # policy forward and sample of a small batch (evaluation panels, C1) and of C3
        dict(name='policy_1k', kind='policy', rows=1024),
        dict(name='policy_c3', kind='policy', rows=65536),
        # the autoregressive head's forward and two-stage sample at C5
        dict(name='policy_ar_c5', kind='policy_ar', rows=262144),
        # one epoch of C4 minibatches over a short rollout, and a small trainer's update
        dict(name='ppo_8k', kind='ppo', steps=16, worlds=8192, minibatch=8192, epochs=1),
        dict(name='ppo_1k', kind='ppo', steps=16, worlds=256, minibatch=1024, epochs=1),
        # C4's advantages
        dict(name='gae_c4', kind='gae', steps=128, worlds=65536),
        # the trainer's rollout (one graph replay: forward, sample, step, buffer writes)
        dict(name='rollout_4k', kind='rollout', steps=16, worlds=4096),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(['env', 'env', 'crowd', 'learn', 'policy', 'policy', 'policy_ar', 'ppo', 'gae', 'rollout'])
    if kind == 'env':
        return dict(kind='env', worlds=_log_int(rng, 256, 65536), monsters=rng.randint(1, 8),
                    rules=rng.choice(['baseline', 'v1', 'reference']), hash=rng.random() < 0.5)
    if kind == 'crowd':
        return dict(kind='env', worlds=_log_int(rng, 256, 65536), monsters=rng.randint(9, 64),
                    rules=rng.choice(['baseline', 'stress', 'reference']), hash=rng.random() < 0.5)
    if kind == 'learn':
        return dict(kind='learn', worlds=_log_int(rng, 256, 65536), maps=rng.choice([1, 4, 32]), clump=rng.randint(0, 1))
    if kind in ('policy', 'policy_ar'):
        return dict(kind=kind, rows=_log_int(rng, 16, 262144))
    if kind == 'ppo':
        mb = 1024 * rng.randint(1, 8)
        steps = rng.choice([8, 16, 32])
        # small minibatches walk apart soonest (see tolerance): few of them
        batches = rng.randint(2, 4) if mb < 4096 else rng.randint(4, 12)
        worlds = mb * batches // steps + rng.randint(0, 31)   # a ragged tail is dropped
        return dict(kind='ppo', steps=steps, worlds=worlds, minibatch=mb, epochs=1)
    if kind == 'gae':
        return dict(kind='gae', steps=_log_int(rng, 8, 256), worlds=_log_int(rng, 64, 65536))
    return dict(kind='rollout', steps=rng.randint(8, 16), worlds=_log_int(rng, 128, 16384))


def _config(case):
    m, rules = case['monsters'], case['rules']
    if rules == 'stress':
        return pkg.make_config(m, hp_lo=40, hp_hi=60, awake_pct=50)
    if rules == 'reference':
        return pkg.reference_config(m)
    if rules == 'v1':
        return pkg.v1_config(m)
    return pkg.baseline_config(m)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _actions(g, rows, worlds):
    """Uniform moves and attacks (C1's stream), [rows, worlds]."""
    return torch.randint(0, 16, (rows, worlds), generator=g, device=DEV, dtype=torch.int64)


def _observations(rows, seed, cfg, steps=24):
    """Observations met `steps` random decisions into an episode, uint8 [rows, 1800]."""
    env = pkg.Env(rows, cfg, seed=seed, device=DEV, hash=False)
    g = _gen(seed + 1)
    for a in _actions(g, steps, rows):
        env.step(a)
    return env.obs.view(rows, -1)


def _ppo_buffer(case, seed):
    """A rollout of the initial policy; rewards, ends and values are C4's draws."""
    T, n = case['steps'], case['worlds']
    env = pkg.Env(n, pkg.baseline_config(), seed=seed, device=DEV, hash=False)
    model = policy.Policy(seed=seed).to(DEV)
    packed = model.packed()
    buf = ppo.RolloutBuffer(T, n, device=DEV)
    value = torch.empty(n, dtype=torch.float32, device=DEV)
    for t in range(T):
        buf.obs[t].copy_(env.obs.view(n, -1))
        policy.policy_fwd_sample(buf.obs[t], *packed, seed, t, buf.actions[t], buf.logp[t], value)
        env.step(buf.actions[t])
    g = _gen(seed + 1)
    hit = torch.rand(T, n, device=DEV, generator=g) < 0.03
    buf.rewards.copy_(torch.where(hit, torch.rand(T, n, device=DEV, generator=g) * 2 - 1, 0.0))
    buf.dones.copy_((torch.rand(T, n, device=DEV, generator=g) < 0.01).to(torch.uint8))
    buf.values.copy_(torch.randn(T, n, device=DEV, generator=g))
    buf.bootstrap.copy_(torch.randn(n, device=DEV, generator=g))
    return buf, model


def _ar_model(seed):
    return policy.ARPolicy(seed=seed).to(DEV).to(torch.bfloat16)


def prepare(case, seed):
    kind = case['kind']
    if kind == 'env':
        n = case['worlds']
        env = pkg.Env(n, _config(case), seed=seed, device=DEV, hash=case['hash'])
        g = _gen(seed + 1)
        for a in _actions(g, 32, n):     # past the first decisions: monsters awake, parts of levels seen
            env.step(a)
        return dict(kind=kind, env=env, actions=_actions(g, RING, n), at=0)
    if kind == 'learn':
        maps = None
        if case['maps'] > 1:
            maps = learn.LearnMaps(pkg.Env(case['maps'], pkg.baseline_config(), seed=seed, device=DEV).floors(), device=DEV)
        env = learn.LearnEnv(case['worlds'], seed=seed, device=DEV, maps=maps, clump=case['clump'])
        for _ in range(32):
            env.step(env.heuristic())
        return dict(kind=kind, env=env)
    if kind == 'policy':
        n = case['rows']
        obs = _observations(n, seed, pkg.baseline_config())
        out = dict(actions=torch.empty(n, dtype=torch.int64, device=DEV), logp=torch.empty(n, device=DEV),
                   value=torch.empty(n, device=DEV), logits=torch.empty((n, 16), device=DEV))
        return dict(kind=kind, obs=obs, packed=policy.Policy(seed=seed).to(DEV).packed(), seed=seed, out=out)
    if kind == 'policy_ar':
        n = case['rows']
        obs = _observations(n, seed, pkg.stress_config(), steps=8)
        out = dict(action=torch.empty(n, dtype=torch.int64, device=DEV), logp=torch.empty(n, device=DEV),
                   value=torch.empty(n, device=DEV), verb_logits=torch.empty((n, 8), device=DEV))
        return dict(kind=kind, obs=obs, packed=_ar_model(seed).packed(), seed=seed, out=out)
    if kind == 'ppo':
        buf, model = _ppo_buffer(case, seed)
        return dict(kind=kind, buf=buf, gen=_gen(seed + 2),
                    ppo=ppo.FastPPO(model, minibatch=case['minibatch'], epochs=case['epochs']))
    if kind == 'gae':
        T, n, g = case['steps'], case['worlds'], _gen(seed)
        hit = torch.rand(T, n, device=DEV, generator=g) < 0.03
        return dict(kind=kind, reward=torch.where(hit, torch.rand(T, n, device=DEV, generator=g) * 2 - 1, 0.0),
                    done=(torch.rand(T, n, device=DEV, generator=g) < 0.01).to(torch.uint8),
                    value=torch.randn(T, n, device=DEV, generator=g), bootstrap=torch.randn(n, device=DEV, generator=g),
                    adv=torch.empty((T, n), device=DEV), returns=torch.empty((T, n), device=DEV))
    if kind == 'rollout':
        env = pkg.Env(case['worlds'], pkg.baseline_config(), seed=seed, device=DEV, hash=False)
        return dict(kind=kind, trainer=train.Trainer(env, policy.Policy(seed=seed).to(DEV), horizon=case['steps'],
                                                     minibatch=1024, seed=seed))
    raise ValueError(kind)


def run(state):
    kind = state['kind']
    if kind == 'env':
        env = state['env']
        obs, out = env.step(state['actions'][state['at'] % RING])
        state['at'] += 1
        res = dict(obs=obs, out=out, state=env.state)
        if env.with_hash:
            res['hash'] = env.hash
        return res
    if kind == 'learn':
        env = state['env']
        actions = env.heuristic()
        obs, out = env.step(actions)
        return dict(actions=actions, obs=obs, mask=env.mask, out=out, state=env.state)
    if kind == 'policy':
        o = state['out']
        policy.policy_fwd_sample(state['obs'], *state['packed'], state['seed'], 5, o['actions'], o['logp'], o['value'],
                                 logits=o['logits'])
        return o
    if kind == 'policy_ar':
        o = state['out']
        policy.policy_fwd_sample_ar(state['obs'], state['packed'], state['seed'], 5, o['action'], o['logp'], o['value'],
                                    verb_logits=o['verb_logits'])
        return o
    if kind == 'ppo':
        terms = state['ppo'].update(state['buf'], generator=state['gen'])
        flat = state['ppo'].flat
        return dict(p=flat.p, m=flat.m, v=flat.v, terms=terms)
    if kind == 'gae':
        adv, returns = policy.gae(state['reward'], state['done'], state['value'], state['bootstrap'], adv=state['adv'],
                                  returns=state['returns'])
        return dict(adv=adv, returns=returns)
    buf = state['trainer'].rollout()
    return dict(obs=buf.obs, actions=buf.actions, logp=buf.logp, values=buf.values, rewards=buf.rewards,
                dones=buf.dones, bootstrap=buf.bootstrap)


def _env_bytes(monsters):
    """One world-step: observation, action, outcome, header and monsters both ways, the view band
    of the level memory both ways, the level bitmap."""
    return 1800 + 8 + 32 + 2 * (24 + 7 * monsters) + 600 + 700


def work(case):
    kind = case['kind']
    if kind == 'env':
        return dict(bytes=case['worlds'] * (_env_bytes(case['monsters']) + (4 if case['hash'] else 0)), flops=0)
    if kind == 'learn':
        return dict(bytes=case['worlds'] * LEARN_BYTES, flops=0)
    if kind == 'policy':
        return dict(bytes=case['rows'] * (1800 + 64 + 4 + 4 + 8) + 2 * POLICY_PARAMS, flops=case['rows'] * TRUNK_FLOPS)
    if kind == 'policy_ar':
        return dict(bytes=case['rows'] * (1800 + 32 + 4 + 4 + 8) + 2 * POLICY_PARAMS, flops=case['rows'] * AR_FLOPS)
    if kind == 'ppo':
        n = case['steps'] * case['worlds']
        steps = n // case['minibatch'] * case['epochs']
        used = steps * case['minibatch']
        # samples gathered, masters and moments both ways once a step, GAE's four arrays
        return dict(bytes=used * (1800 + 8 + 8 + 12) + steps * POLICY_PARAMS * 28 + n * 17, flops=used * PPO_FLOPS)
    if kind == 'gae':
        return dict(bytes=case['steps'] * case['worlds'] * 17 + 4 * case['worlds'], flops=0)
    n = case['steps'] * case['worlds']
    return dict(bytes=n * (_env_bytes(8) + 1800 + 8 + 4 + 4 + 4 + 1), flops=n * TRUNK_FLOPS)


def tolerance(case):
    kind = case['kind']
    if kind in ('env', 'learn'):
        return 'exact'                         # the rules are integer arithmetic, bit for bit
    if kind == 'gae':
        return dict(rel=1e-5)                  # 32-bit sums
    if kind in ('policy', 'policy_ar'):
        # Against torch's bf16 products: single bf16 steps (rel 6e-5, max 7e-3); a draw next to
        # a boundary of the cumulative sum may fall to the neighbour.
        return dict(rel=3e-4, max=5e-2, differ=5e-4)
    if kind == 'ppo':
        # The samples of each minibatch in another order: rel 2e-5 after 16 steps of 8,192 and
        # 2e-3 (max 0.11) after 4 of 1,024; 16 of those walk apart by 5e-2, since Adam's first
        # steps are +-lr for any gradient.
        return dict(rel=1e-2, max=0.5)
    # torch's products in the rollout: no action of 4,096 x 16 changed; one that does changes its
    # world's later rows
    return dict(rel=2e-2, max=0.9, differ=2e-3)


def _relu_trunk(obs, params):
    """h2 of the trunk in 64 bits; params: state dict of 64-bit tensors."""
    h = torch.relu(obs.double() @ params['l1.weight'].t() + params['l1.bias'])
    return torch.relu(h @ params['l2.weight'].t() + params['l2.bias'])


def _doubles(model):
    return {k: v.detach().double() for k, v in model.state_dict().items()}


def _gae64(reward, done, value, bootstrap, gamma=0.99, lam=0.95):
    adv = torch.empty(reward.shape, dtype=torch.float64, device=reward.device)
    nxt, run_ = bootstrap.double(), torch.zeros_like(bootstrap, dtype=torch.float64)
    for t in range(reward.shape[0] - 1, -1, -1):
        live = 1.0 - done[t].double()
        v = value[t].double()
        run_ = reward[t].double() + gamma * nxt * live - v + gamma * lam * live * run_
        adv[t] = run_
        nxt = v
    return adv, adv + value.double()


def exact(case, seed):
    kind = case['kind']
    if kind in ('policy', 'policy_ar'):
        state = prepare(case, seed)
        # the model as it is run: its weights are bf16
        ar = kind == 'policy_ar'
        params = _doubles(_ar_model(seed) if ar else policy.Policy(seed=seed).to(DEV).to(torch.bfloat16))
        outs = []
        for rows in state['obs'].split(16384):
            h = _relu_trunk(rows, params)
            if ar:
                outs.append((h @ params['verb.weight'].t() + params['verb.bias'],
                             (h @ params['value.weight'].t() + params['value.bias']).squeeze(1)))
            else:
                o = h @ params['head.weight'].t() + params['head.bias']
                outs.append((o[:, :16], o[:, 16]))
        logits, value = (torch.cat(x) for x in zip(*outs))
        if ar:
            return dict(action=None, logp=None, value=value, verb_logits=logits)
        return dict(actions=None, logp=None, value=value, logits=logits)
    if kind == 'gae':
        s = prepare(case, seed)
        adv, returns = _gae64(s['reward'], s['done'], s['value'], s['bootstrap'])
        return dict(adv=adv, returns=returns)
    if kind != 'ppo':
        return None
    buf, model = _ppo_buffer(case, seed)
    params = {k: v.clone().requires_grad_() for k, v in _doubles(model).items()}
    m = {k: torch.zeros_like(v) for k, v in params.items()}
    v2 = {k: torch.zeros_like(v) for k, v in params.items()}
    adv, ret = _gae64(buf.rewards, buf.dones, buf.values, buf.bootstrap)
    adv, ret = adv.flatten(), ret.flatten()
    adv = (adv - adv.mean()) / (adv.std() + 1e-8)
    n, mb, gen, step, terms = adv.numel(), case['minibatch'], _gen(seed + 2), 0, None
    obs, actions, logp = buf.obs.view(n, -1), buf.actions.view(n), buf.logp.view(n).double()
    for _ in range(case['epochs']):
        order = torch.randperm(n, device=DEV, generator=gen)
        for at in order[:n // mb * mb].split(mb):
            h = _relu_trunk(obs[at], params)
            out = h @ params['head.weight'].t() + params['head.bias']
            lp = torch.log_softmax(out[:, :16], -1)
            ratio = torch.exp(lp.gather(1, actions[at, None]).squeeze(1) - logp[at])
            pg = -torch.minimum(ratio * adv[at], ratio.clamp(0.8, 1.2) * adv[at]).mean()
            vl = 0.5 * (out[:, 16] - ret[at]).square().mean()
            ent = -(lp.exp() * lp).sum(-1).mean()
            grads = torch.autograd.grad(pg + 0.5 * vl - 0.01 * ent, list(params.values()))
            norm = torch.sqrt(sum(g.square().sum() for g in grads))
            coef, step = torch.clamp(0.5 / (norm + 1e-6), max=1.0), step + 1
            with torch.no_grad():
                for (k, p), g in zip(params.items(), grads):
                    m[k].mul_(0.9).add_(g * coef, alpha=0.1)
                    v2[k].mul_(0.999).add_((g * coef).square(), alpha=0.001)
                    p.sub_(3e-4 / (1 - 0.9 ** step) * m[k] / (torch.sqrt(v2[k] / (1 - 0.999 ** step)) + 1e-5))
            terms = torch.stack([pg, vl, ent]).detach()

    def flat(d):   # segments start on 64-element boundaries
        parts = []
        for k in ('l1.weight', 'l1.bias', 'l2.weight', 'l2.bias', 'head.weight', 'head.bias'):
            x = d[k].detach().reshape(-1)
            parts.append(torch.nn.functional.pad(x, (0, -x.numel() % 64)))
        return torch.cat(parts)
    # the moments of the bf16 path leave those of the 64-bit one step by step (the first by 0.01
    # at once), which says nothing about either: only the weights and the losses are compared
    return dict(p=flat(params), m=None, v=None, terms=terms)
