"""The step kernel (bounded transform, its gradient and a leapfrog update in
one launch) against the torch expressions it stands for: equal bit for bit,
also where the transform saturates, and in the posterior and a leapfrog
trajectory built on it."""
import numpy as np
import pytest
import torch

from forcepho_amd import synth
from forcepho_amd.batch import DeviceSplines, PatchBatch
from forcepho_amd.hmc import HMC, DevicePosterior
from helpers import make_config_patch

pytestmark = pytest.mark.gpu


class TorchPosterior(DevicePosterior):
    """The same posterior through the torch expressions only."""

    def native(self, *vectors):
        return False


def same(a, b):
    return torch.equal(torch.nan_to_num(a), torch.nan_to_num(b)) and \
        torch.equal(torch.isfinite(a), torch.isfinite(b))


# one lane, a wave less one, a wave and one lane, several waves
@pytest.mark.parametrize("n", [1, 63, 65, 4099])
def test_step_equals_torch(hip, n):
    rng = np.random.default_rng(n)
    dev = torch.device("cuda", 0)
    vec = lambda v: torch.as_tensor(v, dtype=torch.float64, device=dev)

    class Stub(DevicePosterior):
        def __init__(self):
            self.lower, self.range = vec(rng.normal(size=n)), vec(10.0 ** rng.uniform(-6, 6, n))
            self.log_range = torch.log(self.range)

    post = Stub()
    z = rng.normal(size=n) * 10.0 ** rng.uniform(-8, 3, n)
    z[:6] = np.array([0.0, -0.0, 800.0, -800.0, np.inf, -np.inf])[:n]
    z, gq, p, g0 = vec(z), *(vec(rng.normal(size=n) * 1e3) for _ in range(3))
    eps, mass = vec(10.0 ** rng.uniform(-6, 0, n)), vec(10.0 ** rng.uniform(-3, 3, n))
    y = torch.sigmoid(z)
    jac = post.range * y * (1.0 - y)
    grad = gq * jac + (1.0 - 2.0 * y)
    a = torch.abs(z)
    lnjac = post.log_range - a - 2.0 * torch.log1p(torch.exp(-a))
    o = {k: torch.full_like(z, 7.0) for k in ("grad", "lnjac", "p_out", "z_out", "q_out")}
    for kick in (1.0, 0.5):
        post.step(z, kick, grad_q=gq, p=p, eps=eps, inv_mass=mass, **o)
        p1 = p + (eps if kick == 1.0 else 0.5 * eps) * grad
        z1 = z + eps * (mass * p1)
        for name, want in dict(grad=grad, lnjac=lnjac, p_out=p1, z_out=z1,
                               q_out=post.lower + torch.sigmoid(z1) * post.range).items():
            assert same(o[name], want), (name, kick)
    post.step(z, q_out=o["q_out"])
    assert same(o["q_out"], post.lower + y * post.range)
    post.step(z, 0.5, grad=g0, p=p, eps=eps, p_out=o["p_out"])
    assert same(o["p_out"], p + 0.5 * eps * g0)


@pytest.mark.parametrize("n_steps", [1, 3])
def test_posterior_and_leapfrog_equal_torch(hip, n_steps):
    patch, scene, theta = make_config_patch(1)
    patch.send_to_device()
    batch = PatchBatch([patch])
    splines = DeviceSplines()
    try:
        lo, hi = synth.theta_bounds(theta, 1)
        got = []
        for cls in (DevicePosterior, TorchPosterior):
            post = cls(batch, splines, lo, hi)
            hmc = HMC(post, post.inverse_transform(theta), step_size=1e-4, n_steps=n_steps, seed=4)
            lnp, grad = post(hmc.z)
            out = [lnp.clone(), grad.clone()]
            p = torch.linspace(-1.0, 1.0, len(theta), dtype=torch.float64, device="cuda")
            out += [v.clone() for v in hmc.leapfrog(hmc.z, p, hmc.grad)]
            hmc.trajectory()
            out += [v.clone() for v in (hmc.z, hmc.lnp, hmc.grad, hmc.accept_prob)]
            assert post.native(hmc.z, p) == (cls is DevicePosterior)
            got.append(out)
        for k, (a, b) in enumerate(zip(*got)):
            assert torch.equal(a, b), k
        # an autograd graph over z is the torch expressions' to build
        assert not DevicePosterior.native(post, hmc.z.clone().requires_grad_())
    finally:
        splines.free()
        batch.free()
        patch.free()
