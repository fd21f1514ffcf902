"""Monsters that cannot move: the crowded step takes their acts together, and finds the ones shut in
by their neighbours with a few row reads at the map's edges and across its 32-column words. Jammed
one- and two-wide corridors along every edge and word boundary, all monsters awake, both RNGs and
REST among the actions: equal to the oracle every step."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from test_env_gpu import compare

pytestmark = pytest.mark.gpu


def corridors():
    f = np.zeros((70, 80), np.uint8)
    f[0, :] = f[69, :] = f[:, 0] = f[:, 79] = 1       # the map's edges
    f[:, 31:33] = f[:, 63:65] = 1                     # across the words of a row
    f[34, :] = 1
    cells = np.zeros_like(f)                          # everyone starts in a few jammed stretches
    for ys, xs in ((slice(0, 1), slice(0, 14)), (slice(69, 70), slice(66, 80)), (slice(28, 35), slice(31, 33)),
                   (slice(0, 14), slice(79, 80)), (slice(58, 70), slice(63, 65)), (slice(40, 52), slice(0, 1))):
        cells[ys, xs] = f[ys, xs]
    return f.reshape(-1), cells.reshape(-1)


def shut_in_count(fields, floor):
    """Awake living monsters, not next to the player, without a free neighbour (numpy)."""
    total = 0
    for w in fields:
        free = floor.reshape(70, 80).astype(bool).copy()
        alive = w['mhp'] > 0
        for p in w['pos'][alive]:
            free[p // 80, p % 80] = False
        py, px = divmod(int(w['player']), 80)
        for p in w['pos'][alive & (w['awake'] > 0)]:
            y, x = divmod(int(p), 80)
            if max(abs(y - py), abs(x - px)) > 1:
                total += not free[max(0, y - 1):y + 2, max(0, x - 1):x + 2].any()
    return total


@pytest.mark.parametrize('count,rng_mode,repair', [(40, 0, 1), (40, 1, 1), (60, 1, 1), (12, 0, 1), (40, 1, 0)])
def test_jammed_corridors_match_oracle(pkg, count, rng_mode, repair):
    print(f'[jammed] count={count} rng={rng_mode} repair={repair}', flush=True)
    cfg = pkg.make_config(count, rng_mode=rng_mode, level_mode=0, awake_pct=100, hp_lo=40, hp_hi=60)
    cfg.repair, cfg.hp = repair, 400                  # episodes long enough for jams to move
    level = corridors()
    n = 24
    gpu = pkg.Env(n, cfg, seed=5, level=level)
    cpu = O.OracleEnv(n, cfg, seed=5, threads=8, level=level)
    compare(gpu, cpu, -1, 'jammed')
    rng = np.random.default_rng(count)
    shut = 0
    for k in range(60):
        a = np.where(rng.random(n) < 0.3, rng.choice([16, 17], n), rng.integers(0, 19, n)).astype(np.int64)
        if k % 10 == 0:
            shut += shut_in_count(gpu.fields(), level[0])
        cpu.step(a)
        gpu.step(torch.from_numpy(a).to(gpu.device))
        compare(gpu, cpu, k, f'jammed{count}')
    assert shut > (20 if count >= 40 else 0)
