"""Which plans take the two-launch route (fpho_launch in include/fpho.h)."""
import numpy as np
import pytest
import torch

from forcepho_amd import synth
from forcepho_amd.batch import PatchBatch
from forcepho_amd.synth import PatchSpec

pytestmark = pytest.mark.gpu


# (exposures, side, factor on the sources' radii, pixels per lane, two launches);
# a source of the synthetic patches reaches 283000 pixels
@pytest.mark.parametrize("n_exp,side,scale,K,two", [
    (1, 32, 1.0, 8, True),
    (16, 256, 1.0, 4, True),       # narrower than the reach
    (2, 1024, 1.0, 8, True),       # 3.7 reaches, 4096 tiles
    (4, 1024, 1.0, 4, False),      # 16384 tiles of them
    (1, 2048, 1.0, 8, False),      # 15 reaches, 8192 tiles
    (8, 512, 1.0, 4, True),        # 0.9 of the reach, 8192 tiles
    (8, 512, 1.0 / 3.0, 4, False)  # 8 reaches
])
def test_wide_exposures_take_one_wave_per_tile(hip, n_exp, side, scale, K, two):
    spec = PatchSpec(n_sources=2, n_bands=1, n_exp_per_band=n_exp, side=side, n_psf=1)
    patch, scene, _ = synth.make_patch(spec, config=64, patch_id=0)
    patch.rad2 = (patch.rad2 * np.float32(scale) ** 2).astype(np.float32)
    patch.send_to_device()
    batch = PatchBatch([patch], launch=dict(pix_per_lane=K, waves_per_group=1, persistent=0))
    try:
        assert batch.two_launches() == two
        batch.set_proposals([scene.get_proposal()])
        batch.evaluate()
        torch.cuda.synchronize()
        want = patch.get_proposer().evaluate_proposal(scene.get_proposal(), patch)[0]
        patch.set_launch(pix_per_lane=K, waves_per_group=1, persistent=0)
        same = patch.get_proposer().evaluate_proposal(scene.get_proposal(), patch)[0]
        assert np.array_equal(batch.chi2_host(0), same)
        assert np.allclose(want, same, rtol=1e-6)
    finally:
        batch.free()
        patch.free()
