"""The GAE kernel at the edges of its split (64 envs a workgroup, one to eight waves of 16 time steps):
bit-equal to the fp32 loop, also where it writes over its inputs; and the normalisation of the
advantages against its elementwise expression."""
import importlib

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (1, 33), (4, 65), (5, 64), (8, 129), (15, 64), (16, 65), (17, 63), (32, 64), (33, 65), (64, 64), (65, 63), (112, 3), (113, 70), (127, 100),
          (128, 64), (129, 1), (144, 64), (145, 9), (300, 130), (512, 7)]


def _draw(T, n):
    g = torch.Generator().manual_seed(1000 * T + n)
    r = torch.rand(T, n, generator=g) * 2 - 1
    d = (torch.rand(T, n, generator=g) < 0.05).to(torch.uint8)
    return r, d, torch.randn(T, n, generator=g), torch.randn(n, generator=g)


def _loop(r, d, v, boot, gamma=0.99, lam=0.95):
    f = np.float32
    r, v, live = r.numpy(), v.numpy(), (1 - d.numpy().astype(f)).astype(f)
    g, gl = f(gamma), f(gamma * lam)
    adv, nxt, acc = np.empty_like(r), boot.numpy(), np.zeros(r.shape[1], f)
    for t in reversed(range(r.shape[0])):
        delta = (r[t] + (g * nxt) * live[t]) - v[t]
        acc = delta + (gl * live[t]) * acc
        adv[t], nxt = acc, v[t]
    return torch.from_numpy(adv), torch.from_numpy(adv + v)


@pytest.mark.parametrize('T,n', SHAPES)
def test_gae_is_the_fp32_loop_bit_for_bit(T, n):
    pol = importlib.import_module('dcss-auto_amd.policy')
    print(f'[gae] T={T} n={n}', flush=True)
    r, d, v, boot = _draw(T, n)
    want, wret = _loop(r, d, v, boot)
    guard = torch.full((T * n + 64,), 7.0, device='cuda')
    adv, ret = pol.gae(r.cuda(), d.cuda(), v.cuda(), boot.cuda(), adv=guard[:T * n].view(T, n))
    assert torch.equal(adv.cpu(), want) and torch.equal(ret.cpu(), wret)
    assert bool((guard[T * n:] == 7.0).all())
    for over in ('reward', 'value'):   # written over an input
        rc, vc = r.cuda(), v.cuda()
        adv, ret = pol.gae(rc, d.cuda(), vc, boot.cuda(), adv=rc if over == 'reward' else vc)
        assert torch.equal(adv.cpu(), want) and torch.equal(ret.cpu(), wret), over


@pytest.mark.parametrize('n', [1, 3, 4, 5, 1023, 1025, 2048 * 1024 + 7])
@pytest.mark.parametrize('shift', [0, 1])
def test_normalisation_is_the_elementwise_expression(n, shift):
    """Bit for bit, with and without 16-byte alignment (one float4 a lane, a tail, more groups than
    the grid); one value and non-finite values normalise to NaN as the expression does."""
    pol = importlib.import_module('dcss-auto_amd.policy')
    g = torch.Generator(device='cuda').manual_seed(n)
    buf = torch.full((n + 8,), 3.0, device='cuda')
    for kind in ('plain', 'nan', 'inf'):
        adv = buf[shift:shift + n]
        adv.copy_(torch.randn(n, generator=g, device='cuda') * 3 + 1)
        if kind != 'plain':
            adv[n // 2] = float(kind)
        want = (adv - adv.mean()) / (adv.std() + 1e-8)
        pol.normalize_(adv)
        assert torch.equal(adv.isnan(), want.isnan()) and torch.equal(adv.nan_to_num(), want.nan_to_num()), kind
        assert bool((buf[shift + n:] == 3.0).all())
        assert (kind == 'plain' and n > 1) or bool(adv.isnan().all())
