"""A NUTS leaf is one leapfrog step, whatever the number of steps of the HMC
trajectories of the same object and however its ``leapfrog`` is overridden
(host, CPU tensors)."""
import numpy as np
import torch

from forcepho_amd.nuts import NUTS
from test_nuts import GaussianPatches


class Counting(NUTS):
    calls = 0

    def leapfrog(self, z, p, grad, eps=None):
        self.calls += 1
        return super().leapfrog(z, p, grad, eps)


def test_nuts_leaf_is_one_leapfrog_step():
    rng = np.random.default_rng(3)
    post = GaussianPatches([np.diag(1.0 + rng.random(3)), np.diag(1.0 + rng.random(2))])
    z = torch.as_tensor(rng.normal(size=5))
    s = Counting(post, z, step_size=0.1, seed=2)
    s.n_steps = 4
    p, eps = torch.as_tensor(rng.normal(size=5)), s.eps
    lnp, grad = post(z)
    p1 = p + 0.5 * eps * grad
    z1 = z + eps * (s.inv_mass * p1)
    lnp1, grad1 = post(z1)
    want = z1, p1 + 0.5 * eps * grad1, lnp1, grad1
    n = post.n_evals
    for a, b in zip(s._leapfrog1(z, p, grad, eps), want):
        assert torch.equal(a, b)
    assert post.n_evals == n + 1 and s.calls == 0
    # and the trajectory of the same object takes its four steps
    s.leapfrog(z, p, grad, eps)
    assert post.n_evals == n + 5
