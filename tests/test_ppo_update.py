"""The host side of FastPPO's update and of the trainer's rollout, without a GPU: the kernels' wrappers are
replaced by checks of what they would be given."""
import importlib

import pytest
import torch

ppo = importlib.import_module('dcss-auto_amd.ppo')


@pytest.fixture
def fast(monkeypatch):
    """A FastPPO of 1,024-sample minibatches without its device buffers; GAE writes its step numbers and
    fails where its output would run past the tensor that it is given."""
    def gae(reward, done, value, bootstrap, gamma, lam, adv=None, returns=None):
        for x in (adv, returns):
            assert x.dtype == torch.float32 and x.is_contiguous() and x.numel() >= reward.numel()
            x.view(-1)[:reward.numel()] = torch.arange(reward.numel(), dtype=torch.float32)
        return adv, returns

    monkeypatch.setattr(ppo.P, 'gae', gae)
    monkeypatch.setattr(ppo.P, 'normalize_', lambda adv: adv.add_(0.5))
    f = ppo.FastPPO.__new__(ppo.FastPPO)
    f.gamma, f.lam, f.dev = 0.99, 0.95, torch.device('cpu')
    return f


def test_advantages_are_sized_by_the_rewards(fast):
    """Rewards of more steps than T: the outputs hold all of them, and given ones that do not are refused."""
    buf = ppo.RolloutBuffer(4, 6, device='cpu')
    for name in ('rewards', 'values', 'dones'):
        setattr(buf, name, torch.cat([getattr(buf, name)] * 2))
    adv, ret = fast.advantages(buf)
    assert torch.equal(ret, torch.arange(48.)) and torch.equal(adv, ret + 0.5)
    full = torch.empty(48)
    for bad in (torch.empty(24), torch.empty(96)[::2], torch.empty(48, dtype=torch.float64)):
        for args in ((bad, full), (full, bad)):
            with pytest.raises(ValueError):
                fast.advantages(buf, *args)


@pytest.mark.parametrize('given', [(), ('adv',), ('ret',), ('adv', 'ret')])
def test_advantages_and_returns_are_each_made_when_not_given(fast, given):
    buf = ppo.RolloutBuffer(4, 6, device='cpu')
    out = {k: torch.empty(24) for k in given}
    adv, ret = fast.advantages(buf, **out)
    assert torch.equal(ret, torch.arange(24.)) and torch.equal(adv, ret + 0.5)
    assert all(x is out[k] for k, x in (('adv', adv), ('ret', ret)) if k in given)


class _Graph:
    replays = 0

    def replay(self):
        self.replays += 1


def _ready(f, buf, graph):
    """What update() finds after construction, and with graph=True after a capture."""
    n = buf.T * buf.N
    f.minibatch, f.epochs, f.graph, f.graph_steps = 1024, 3, graph, 16
    f.perm, f._packed, f.head_out, f._args_key, f._g, f._g_buf, f._adv = None, True, None, None, None, None, None
    f.cursor, f.step_t, f.loss_parts = torch.zeros(2, dtype=torch.int32), torch.zeros(3), torch.zeros(128)
    f.seen = []
    f._struct = lambda *a: None
    f._step = lambda obs, actions, logp, adv, ret: f.seen.append((adv.clone(), ret.clone(), f.perm.clone()))

    def capture(b):
        if f._adv is None or f._adv.numel() != n:
            f._adv, f._ret = torch.zeros(n), torch.zeros(n)
        if f.perm is None or f.perm.shape != (n,):
            f.perm = torch.zeros(n, dtype=torch.int64)
        f._g, f._g_buf = _Graph(), b
        f._g.reads = [x.data_ptr() for x in (f.perm, b.obs, b.actions, b.logp)]
        f._g_key = f._key(*f._views(b), f._adv, f._ret)
    f._capture = capture


@pytest.mark.parametrize('graph', [False, True])
@pytest.mark.parametrize('where', ['subclass', 'instance', 'class'])
def test_update_calls_a_replaced_advantages_with_the_buffer_alone(fast, monkeypatch, graph, where):
    buf = ppo.RolloutBuffer(4, 512, device='cpu')
    mine = torch.randn(2048), torch.randn(2048)

    def advantages(self, b):
        assert b is buf
        return mine
    _ready(fast, buf, graph)
    if where == 'subclass':
        fast.__class__ = type('Own', (ppo.FastPPO,), dict(advantages=advantages))
    elif where == 'instance':
        fast.advantages = lambda b: advantages(fast, b)
    else:
        monkeypatch.setattr(ppo.FastPPO, 'advantages', advantages)
    fast.update(buf, generator=torch.Generator().manual_seed(1))
    if graph:
        assert fast._g.replays == 3 and torch.equal(fast._adv, mine[0]) and torch.equal(fast._ret, mine[1])
    else:
        assert len(fast.seen) == 6 and all(torch.equal(a, mine[0]) and torch.equal(r, mine[1]) for a, r, _ in fast.seen)


@pytest.mark.parametrize('graph', [False, True])
def test_a_replaced_set_order_may_keep_the_orders_it_is_given(fast, graph):
    """The same orders as randperm draws from the generator, each in a tensor of its own."""
    buf = ppo.RolloutBuffer(4, 512, device='cpu')
    _ready(fast, buf, graph)
    kept, orig = [], fast.set_order

    def set_order(perm):
        kept.append(perm)
        orig(perm)
    fast.set_order = set_order
    fast.update(buf, generator=torch.Generator().manual_seed(5))
    g = torch.Generator().manual_seed(5)
    assert len(kept) == 3 and all(torch.equal(k, torch.randperm(2048, generator=g)) for k in kept)
    assert torch.equal(fast.perm, kept[-1])


def test_update_captures_again_when_the_graph_holds_other_buffers(fast):
    """An order of another size between two updates, and a replaced tensor of the buffer: the captured
    launches would read the old allocations."""
    buf = ppo.RolloutBuffer(4, 512, device='cpu')
    _ready(fast, buf, True)

    def update():
        fast.update(buf, generator=torch.Generator().manual_seed(1))
        assert fast._g.reads == [x.data_ptr() for x in (fast.perm, buf.obs, buf.actions, buf.logp)]
        return fast._g
    first, old_perm = update(), fast.perm
    assert update() is first                      # nothing changed: the same graph
    fast.set_order(torch.arange(1024))
    second = update()
    assert second is not first and fast.perm is not old_perm and fast.perm.shape == (2048,)
    old_logp, buf.logp = buf.logp, buf.logp.clone()
    assert update() is not second and old_logp is not buf.logp
    fast.set_order(torch.arange(2048).view(2, 1024))   # as many values in another shape
    update()
    assert fast.perm.shape == (2048,)


@pytest.mark.parametrize('where', ['instance', 'class', None])
def test_rollout_steps_through_a_replaced_step(pkg, monkeypatch, where):
    """Env.step wrapped on the instance or on the class (to count or log steps) sees every step; the
    class as it is goes through step_into."""
    train = importlib.import_module('dcss-auto_amd.train')
    monkeypatch.setattr(train.P, 'policy_fwd_sample', lambda *a, **k: None)
    monkeypatch.setattr(train.P, 'policy_fwd', lambda *a, **k: None)
    calls = []
    env = pkg.Env.__new__(pkg.Env)
    env.out = torch.zeros(6, 8)
    monkeypatch.setattr(pkg.Env, 'step_into', lambda self, *a: calls.append('step_into'))
    if where == 'instance':
        env.step = lambda actions, obs: calls.append('step')
    elif where == 'class':
        monkeypatch.setattr(pkg.Env, 'step', lambda self, actions, obs: calls.append('step'))
    t = train.Trainer.__new__(train.Trainer)
    t.buf, t.env, t.T, t.seed = ppo.RolloutBuffer(4, 6, device='cpu'), env, 4, 1
    t.bias, t.wpk, t.logits = (None, None, None), None, None
    t.t_dev, t.next_obs = torch.zeros(1, dtype=torch.int32), torch.zeros(6, 1800, dtype=torch.uint8)
    t._rollout_body()
    assert calls == ['step' if where else 'step_into'] * 4


def test_update_refuses_rewards_of_another_size_than_the_graph(fast):
    """The captured advantages hold T x N values."""
    buf = ppo.RolloutBuffer(4, 512, device='cpu')
    _ready(fast, buf, True)
    fast.update(buf, generator=torch.Generator().manual_seed(1))
    for name in ('rewards', 'values', 'dones'):
        setattr(buf, name, torch.cat([getattr(buf, name)] * 2))
    with pytest.raises(ValueError):
        fast.update(buf, generator=torch.Generator().manual_seed(1))
