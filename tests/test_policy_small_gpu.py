"""The small-batch policy kernels against the large-batch one: every row's outputs are the same
bits whatever batch it is in (the kernels share the packed weights, the contraction order and
the accumulation order), at the tile edges of the 32- and 64-sample workgroups and at both
sides of the batch sizes where the dispatch changes."""
import importlib

import pytest
import torch

pytestmark = pytest.mark.gpu

BIG = 20000   # a batch of the 256-sample kernel
SIZES = [1, 31, 32, 33, 64, 1000, 8191, 8192, 8193, 8193 + 63, 16383, 16384, 16385]


def _obs(n, seed):
    """Rows of every byte value, among them all-zero and all-255 ones; an 8-byte aligned view."""
    g = torch.Generator(device='cuda').manual_seed(seed)
    raw = torch.zeros(8 + n * 1800, dtype=torch.uint8, device='cuda')
    obs = raw[8:].view(n, 1800)
    obs.copy_(torch.randint(0, 256, (n, 1800), generator=g, device='cuda', dtype=torch.uint8))
    obs[0] = 0
    obs[n // 2] = 255
    return obs


@pytest.mark.parametrize('M', SIZES)
def test_small_batches_equal_the_large_kernel(M):
    pol = importlib.import_module('dcss-auto_amd.policy')
    print(f'[policy_small] M={M}', flush=True)
    obs = _obs(BIG, 3)
    g = torch.Generator().manual_seed(4)
    model = pol.Policy(seed=5)
    ar = pol.ARPolicy(seed=6)
    with torch.no_grad():   # biases of the weights' scale: a misplaced one moves the outputs
        for layer in (model.l1, model.l2, model.head, ar.l1, ar.l2, ar.verb, ar.value, ar.t1, ar.t2):
            layer.bias.copy_(torch.randn(layer.bias.shape, generator=g) * 0.1)
    packed = model.cuda().packed()
    apacked = ar.cuda().to(torch.bfloat16).packed()

    def outputs(rows):
        n = rows.shape[0]
        f = lambda *s: torch.full(s, float('nan'), device='cuda')
        i = lambda dt: torch.full((n + 1,), -7, dtype=dt, device='cuda')   # one guard row
        act, lp, val, lg = i(torch.int64), f(n + 1), f(n + 1), f(n + 1, 16)
        pol.policy_fwd_sample(rows, *packed, 9, 3, act[:n], lp[:n], val[:n], logits=lg[:n])
        lg0, val0 = pol.policy_fwd(rows, *packed)
        a2, lp2, v2, vb, tg = i(torch.int64), f(n + 1), f(n + 1), i(torch.int32), i(torch.int32)
        vl, tl = f(n + 1, 8), f(n + 1, 25)
        pol.policy_fwd_sample_ar(rows, apacked, 9, 3, a2[:n], lp2[:n], v2[:n], verb=vb[:n], target=tg[:n],
                                 verb_logits=vl[:n], target_logits=tl[:n])
        for x in (act, lp, val, lg, a2, lp2, v2, vb, tg, vl, tl):   # nothing past the batch
            guard = x[n:]
            assert bool(torch.isnan(guard).all() if x.is_floating_point() else (guard == -7).all())
        return [x[:M] for x in (act, lp, val, lg, lg0, val0, a2, lp2, v2, vb, tg, vl, tl)]

    for k, (small, big) in enumerate(zip(outputs(obs[:M]), outputs(obs))):
        assert torch.equal(small, big), f'output {k}'
