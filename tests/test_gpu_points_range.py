"""Point values of wide nets in batches that hold points outside the split
contraction's range (coordinates above 1e6, infinite, NaN): each point has the value it
has alone, within 1e-4 of its magnitude of float64 where that is finite, and such a batch
costs about what its points cost, not a workgroup's time for each of them."""
import numpy as np
import pytest
import torch

from oracle import mlp as omlp
from niq import implicit_mlp_utils, models

pytestmark = pytest.mark.gpu


def batch(n, share, seed):
    rng = np.random.default_rng(seed)
    x = rng.uniform(-1, 1, size=(n, 3)).astype(np.float32)
    odd = np.flatnonzero(rng.random(n) < share)
    kinds = np.array([[2e6, -3e6, 5e7], [np.nan, 0, 0], [0, np.inf, 1], [1, -2e6, 0.5]], np.float32)
    x[odd] = kinds[np.arange(odd.size) % 4]
    return x, odd


@pytest.mark.parametrize("hidden,act", [([256, 256], "relu"), ([250, 256], "tanh"), ([512, 512], "relu")])
@pytest.mark.parametrize("n,share", [(1, 1.0), (63, 1.0), (64, 0.5), (65, 0.9), (1000, 1.0), (5000, 0.02), (40000, 0.5),
                                     (40001, 0.98)])
def test_mixed_batch_has_each_points_own_value(hidden, act, n, share):
    p = models.random_mlp(hidden, activation=act, init="xavier", seed=4)
    f, _ = implicit_mlp_utils.implicit_from_params(p, "affine_fixed")
    x, odd = batch(n, share, seed=n)
    got = f(p, torch.as_tensor(x, device="cuda")).cpu().numpy()
    plain = np.setdiff1d(np.arange(n), odd)
    if plain.size:   # the points inside the range by themselves
        alone = f(p, torch.as_tensor(x[plain], device="cuda")).cpu().numpy()
        assert np.array_equal(got[plain], alone)
    for q in range(min(4, odd.size)):   # the others: one value for each of the four kinds
        same = got[odd[q::4]]
        alone = f(p, torch.as_tensor(x[odd[q]][None], device="cuda")).cpu().numpy()
        assert np.array_equal(same, np.broadcast_to(alone, same.shape), equal_nan=True)
    fin = np.isfinite(x).all(axis=1)
    r64 = omlp.eval_points(p, x[fin], np.float64).reshape(-1)
    scale = np.maximum(1.0, np.abs(x[fin]).max(axis=1, initial=0.0))
    assert np.all(np.abs(got[fin] - r64) <= 1e-4 * scale)


def test_points_outside_the_range_cost_what_points_cost():
    p = models.random_mlp([512] * 3, seed=5)
    f, _ = implicit_mlp_utils.implicit_from_params(p, "affine_fixed")
    ms = {}
    for share in (0.0, 0.5, 1.0):
        x = torch.as_tensor(batch(100000, share, seed=1)[0], device="cuda")
        f(p, x)
        e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        e[0].record()
        for _ in range(3):
            f(p, x)
        e[1].record()
        torch.cuda.synchronize()
        ms[share] = e[0].elapsed_time(e[1])
    print(ms, flush=True)
    # the FP32 contraction takes 1.7 times the split one's time
    assert ms[0.5] < 4 * ms[0.0] and ms[1.0] < 4 * ms[0.0]
