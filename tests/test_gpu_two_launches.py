"""The two-launch pixel pass (one wave per 64-pixel slot, then one per (tile,
source)), which small plans take, against one wave per tile, which the
zero-allocation entry point keeps: equal bit for bit at every tile size and
precision mode, on exposures whose last tile, slot and Gaussian block are
partly filled."""
import ctypes
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest
import torch

from forcepho_amd import _lib, synth
from forcepho_amd.limits import source_struct_dtype
from forcepho_amd.synth import PatchSpec
from helpers import oracle_render, proposal_for

pytestmark = pytest.mark.gpu

SPECS = {
    # one slot, one source, fewer Gaussians than a wave
    "one_slot": PatchSpec(n_sources=1, n_bands=1, n_exp_per_band=1, side=8, n_psf=1),
    # two slots, the second mostly padding; 64 and 128 Gaussians exactly
    "padded": PatchSpec(n_sources=2, n_bands=2, n_exp_per_band=[1, 2], side=9, n_psf=[4, 7]),
    # more than 64 Gaussians of one source, masked pixels, ragged superpixels
    "wide_psf": PatchSpec(n_sources=3, n_bands=1, n_exp_per_band=2, side=45, n_psf=8,
                          mask_frac=0.2, psf_elliptical=True, psf_per_exposure=True),
    # sources on one side of a large exposure: slots that no Gaussian meets
    "uneven": PatchSpec(n_sources=9, n_bands=2, n_exp_per_band=[3, 1], side=101, n_psf=[3, 6],
                        dither=1.5),
}


@pytest.mark.parametrize("K", [1, 2, 4, 8])
@pytest.mark.parametrize("name", sorted(SPECS))
def test_two_launches_equal_one_wave_per_tile(hip, name, K):
    spec = SPECS[name]
    patch, scene, theta = synth.make_patch(spec, config=61, patch_id=len(name),
                                           return_residual=True, render=oracle_render)
    patch.send_to_device()
    try:
        nb, ns = len(patch.band_N), int(patch.n_sources)
        prop = proposal_for(scene, synth.make_proposals(theta, nb, 1, config=61)[0])
        prop_dev = torch.from_numpy(np.ascontiguousarray(prop, dtype=source_struct_dtype)
                                    .view(np.uint8).copy()).cuda()
        stream = ctypes.c_void_p(int(torch.cuda.current_stream().cuda_stream))
        lib = _lib.lib()
        for cull in (1, 0):
            patch.set_launch(pix_per_lane=K, waves_per_group=2, persistent=0, cull=cull)
            for mode in ("mixed", "mixed_centre", "fp64_reduce", "fp32"):
                patch.set_precision(mode)
                print(name, "K", K, "cull", cull, mode, flush=True)
                got = []
                for fn in (lib.fpho_evaluate_async, lib.fpho_evaluate_async_noalloc):
                    chi2 = torch.full((nb,), 7.0, dtype=torch.float64, device="cuda")
                    dchi2 = torch.full((nb * ns * 7,), 7.0, dtype=torch.float64, device="cuda")
                    _lib.check(fn(patch.device_patch, _lib.dptr(prop_dev), _lib.dptr(chi2),
                                  _lib.dptr(dchi2), stream))
                    torch.cuda.synchronize()
                    got.append((chi2.cpu().numpy(), dchi2.cpu().numpy(),
                                patch.retrieve_array("residual")))
                for a, b in zip(*got):
                    assert np.all(np.isfinite(a)) and np.array_equal(a, b), (cull, mode)
    finally:
        patch.free()


def _evaluators(patch, scene, theta):
    nb, ns = len(patch.band_N), int(patch.n_sources)
    prop = proposal_for(scene, synth.make_proposals(theta, nb, 1, config=61)[0])
    prop_dev = torch.from_numpy(np.ascontiguousarray(prop, dtype=source_struct_dtype)
                                .view(np.uint8).copy()).cuda()
    chi2 = torch.full((nb,), 7.0, dtype=torch.float64, device="cuda")
    dchi2 = torch.full((nb * ns * 7,), 7.0, dtype=torch.float64, device="cuda")

    def stream_ordered():
        stream = ctypes.c_void_p(int(torch.cuda.current_stream().cuda_stream))
        _lib.check(_lib.lib().fpho_evaluate_async(patch.device_patch, _lib.dptr(prop_dev),
                                                  _lib.dptr(chi2), _lib.dptr(dchi2), stream))

    proposer = patch.get_proposer()
    return lambda: proposer.evaluate_proposal(prop, patch)[:2], stream_ordered, chi2, dchi2


def test_capture_after_synchronous_evaluations_only(hip):
    # the plan has no workspace of its own then and none may be allocated
    patch, scene, theta = synth.make_patch(SPECS["uneven"], config=61, patch_id=6,
                                           return_residual=False, render=oracle_render)
    patch.send_to_device()
    try:
        sync, stream_ordered, chi2, dchi2 = _evaluators(patch, scene, theta)
        want = sync()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            stream_ordered()
        for _ in range(3):
            chi2.fill_(7.0)
            dchi2.fill_(7.0)
            graph.replay()
            torch.cuda.synchronize()
            assert np.array_equal(chi2.cpu().numpy(), want[0])
            assert np.array_equal(dchi2.cpu().numpy().astype(np.float32),
                                  np.asarray(want[1]).reshape(-1))
            assert np.array_equal(sync()[0], want[0])
        stream_ordered()   # with a workspace of its own
        torch.cuda.synchronize()
        assert np.array_equal(chi2.cpu().numpy(), want[0])
    finally:
        patch.free()


def test_threads_share_the_synchronous_workspace(hip):
    patches, calls = [], []
    try:
        for i, name in enumerate(("padded", "uneven", "wide_psf")):
            patch, scene, theta = synth.make_patch(SPECS[name], config=61, patch_id=i,
                                                   return_residual=False, render=oracle_render)
            patch.send_to_device()
            patches.append(patch)
            calls.append(_evaluators(patch, scene, theta)[0])
        want = [call() for call in calls]
        with ThreadPoolExecutor(len(calls)) as pool:
            got = list(pool.map(lambda call: [call() for _ in range(20)], calls))
        for w, results in zip(want, got):
            for r in results:
                assert np.array_equal(r[0], w[0]) and np.array_equal(r[1], w[1])
    finally:
        for patch in patches:
            patch.free()
