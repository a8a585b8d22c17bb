"""Point values of TanH and ELU nets, whose point pass is compiled for that activation
alone, against the float32 oracle: within 1e-5 * max |oracle32| (the parity suite's
bar), and the same bits for a batch and for its parts (ragged tiles)."""
import numpy as np
import pytest
import torch

from oracle import mlp as omlp
from niq import implicit_mlp_utils, models

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("act,init", [("tanh", "xavier"), ("elu", "he")])
@pytest.mark.parametrize("hidden", [[32, 20], [64] * 3, [128, 100], [200, 130]])
def test_points_of_one_activation(act, init, hidden):
    p = models.random_mlp(hidden, activation=act, init=init, seed=hidden[0])
    f, _ = implicit_mlp_utils.implicit_from_params(p, "affine_fixed")
    x = np.random.default_rng(1).uniform(-1, 1, (1003, 3)).astype(np.float32)
    xd = torch.as_tensor(x, device="cuda")
    got = f(p, xd)
    want = omlp.eval_points(p, x, np.float32).reshape(-1)
    assert np.abs(got.cpu().numpy() - want).max() <= 1e-5 * np.abs(want).max()
    for n in (1, 15, 64, 65):
        assert torch.equal(f(p, xd[:n]), got[:n]), n
