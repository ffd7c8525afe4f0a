"""When a posterior takes the step kernel: never on a gradient that is not the
batch's own buffer, nor on a vector whose memory does not hold its values."""
import pytest
import torch

from forcepho_amd import synth
from forcepho_amd.batch import DeviceSplines, PatchBatch
from forcepho_amd.hmc import HMC, DevicePosterior
from helpers import make_config_patch

pytestmark = pytest.mark.gpu


class Strided(PatchBatch):
    """Hands out its gradient as every second element of a buffer."""

    def lnlike_and_grad(self, theta, splines, stream=None):
        ll, g = super().lnlike_and_grad(theta, splines, stream)
        return ll, torch.stack([g, torch.zeros_like(g)], dim=1).reshape(-1)[::2]


def wrapped(batch):
    inner = batch.lnlike_and_grad

    def lnlike_and_grad(theta, splines, stream=None):
        ll, g = inner(theta, splines, stream)
        return ll, torch.stack([g, torch.zeros_like(g)], dim=1).reshape(-1)[::2]

    batch.lnlike_and_grad = lnlike_and_grad
    return batch


@pytest.fixture(scope="module")
def target(hip):
    patch, scene, theta = make_config_patch(1)
    patch.send_to_device()
    splines = DeviceSplines()
    yield patch, splines, theta, synth.theta_bounds(theta, 1)
    splines.free()
    patch.free()


def results(batch, splines, theta, bounds, z_of=lambda z: z):
    post = DevicePosterior(batch, splines, *bounds)
    hmc = HMC(post, post.inverse_transform(theta), step_size=1e-4, n_steps=2, seed=4)
    p = torch.linspace(-1.0, 1.0, len(theta), dtype=torch.float64, device="cuda")
    z = z_of(hmc.z)
    return post.native(z), [v.clone() for v in hmc.leapfrog(z, p, hmc.grad) + post(z)]


def test_gradients_of_an_overridden_batch(target):
    patch, *rest = target
    batches = [c([patch]) for c in (PatchBatch, Strided, PatchBatch)]
    wrapped(batches[2])
    try:
        native, out = zip(*(results(b, *rest) for b in batches))
        assert native == (True, False, False)
        for vectors in zip(*out):
            assert torch.equal(vectors[0], vectors[1]) and torch.equal(vectors[0], vectors[2])
    finally:
        for b in batches:
            b.free()


def test_negated_view(target):
    patch, *rest = target
    batch = PatchBatch([patch])
    try:
        _, want = results(batch, *rest)
        native, got = results(batch, *rest, z_of=lambda z: torch._neg_view(-z))
        assert not native
        for a, b in zip(got, want):
            assert torch.equal(a, b)
    finally:
        batch.free()
