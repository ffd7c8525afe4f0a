"""The workspace of the two-launch pixel pass: when it is asked for, and what
happens where it is not to be had."""
import ctypes

import numpy as np
import pytest
import torch

from forcepho_amd import _lib, synth
from forcepho_amd.limits import source_struct_dtype
from forcepho_amd.synth import PatchSpec
from helpers import oracle_render, proposal_for

pytestmark = pytest.mark.gpu

SPEC = PatchSpec(n_sources=5, n_bands=2, n_exp_per_band=[2, 1], side=61, n_psf=3)


def test_first_stream_ordered_call_beside_a_capture(hip):
    """A patch evaluated synchronously so far is evaluated on one stream while
    another captures in global mode (torch's): the capture stays valid."""
    patch, scene, theta = synth.make_patch(SPEC, config=63, patch_id=0, render=oracle_render)
    patch.send_to_device()
    try:
        prop = np.ascontiguousarray(proposal_for(scene, theta), dtype=source_struct_dtype)
        want = patch.get_proposer().evaluate_proposal(prop, patch)
        prop_dev = torch.from_numpy(prop.view(np.uint8).copy()).cuda()
        chi2 = torch.full((2,), 7.0, dtype=torch.float64, device="cuda")
        dchi2 = torch.full((2 * 5 * 7,), 7.0, dtype=torch.float64, device="cuda")
        x = torch.arange(8.0, device="cuda")
        beside = torch.cuda.Stream()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = x * 2.0
            _lib.check(_lib.lib().fpho_evaluate_async(
                patch.device_patch, _lib.dptr(prop_dev), _lib.dptr(chi2), _lib.dptr(dchi2),
                ctypes.c_void_p(int(beside.cuda_stream))))
            y = y + 1.0
        torch.cuda.synchronize()
        assert np.array_equal(chi2.cpu().numpy(), want[0])
        assert np.array_equal(dchi2.cpu().numpy().astype(np.float32), want[1].reshape(-1))
        for step in range(3):
            x.fill_(float(step))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.all(y == 2.0 * step + 1.0)
    finally:
        patch.free()
