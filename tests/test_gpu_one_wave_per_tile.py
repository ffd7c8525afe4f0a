"""The one-wave-per-tile kernels at every launch shape that set_launch offers,
against the two launches: small plans reach them through the zero-allocation
entry point only.  Equal bit for bit, also where the Gaussians of an exposure
outnumber the slot masks and activity words that the kernels keep in LDS."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from forcepho_amd import _lib, synth
from forcepho_amd.limits import source_struct_dtype
from forcepho_amd.synth import PatchSpec
from helpers import CHI2_RTOL, chi2_relerr, grad_mismatch, oracle_render

pytestmark = pytest.mark.gpu

MASK_CAP, ACT_CAP = 6144, 65536   # kMaskCapMax and 64 kActWordsMax of csrc/kernels.h


def routes(patch, prop, launch, mode):
    """chi2, dchi2 [bands, sources, 7] and residual: two launches, one wave per tile."""
    patch.set_launch(**launch)
    patch.set_precision(mode)
    nb, ns = len(patch.band_N), int(patch.n_sources)
    prop_dev = torch.from_numpy(np.ascontiguousarray(prop, dtype=source_struct_dtype)
                                .view(np.uint8).copy()).cuda()
    stream = ctypes.c_void_p(int(torch.cuda.current_stream().cuda_stream))
    lib, out = _lib.lib(), []
    for fn in (lib.fpho_evaluate_async, lib.fpho_evaluate_async_noalloc):
        chi2 = torch.full((nb,), 7.0, dtype=torch.float64, device="cuda")
        dchi2 = torch.full((nb * ns * 7,), 7.0, dtype=torch.float64, device="cuda")
        _lib.check(fn(patch.device_patch, _lib.dptr(prop_dev), _lib.dptr(chi2),
                      _lib.dptr(dchi2), stream))
        torch.cuda.synchronize()
        out.append((chi2.cpu().numpy(), dchi2.cpu().numpy().reshape(nb, ns, 7),
                    patch.retrieve_array("residual")))
    return out


def make(spec, patch_id, render=oracle_render):
    patch, scene, _ = synth.make_patch(spec, config=65, patch_id=patch_id,
                                       return_residual=True, render=render)
    patch.send_to_device()
    return patch, scene.get_proposal()


@pytest.fixture(scope="module")
def ragged(hip):
    # more tiles than the workgroups of one CU at K = 1, a last tile and slot
    # that are partly filled, and a whole number of 64-Gaussian blocks (576) in the second
    specs = [PatchSpec(n_sources=7, n_bands=2, n_exp_per_band=[3, 1], side=101, n_psf=[3, 5]),
             PatchSpec(n_sources=64, n_bands=1, n_exp_per_band=2, side=40, n_psf=1)]
    patches = [make(s, i) for i, s in enumerate(specs)]
    counts = [int(p.n_sources) * int(n) for p, _ in patches for n in p.n_psf_per_source]
    assert counts == [189, 315, 576] and 576 % 64 == 0
    yield patches
    for p, _ in patches:
        p.free()


@pytest.mark.parametrize("persistent", [0, 1])
@pytest.mark.parametrize("W", [1, 2, 3, 4])
@pytest.mark.parametrize("K", [1, 2, 4, 8])
def test_every_launch_shape_equals_the_two_launches(ragged, K, W, persistent):
    for patch, prop in ragged:
        for mode in ("mixed", "mixed_centre", "fp64_reduce"):
            for cull in (1, 0):
                launch = dict(pix_per_lane=K, waves_per_group=W, persistent=persistent,
                              groups_per_cu=4, cull=cull)
                print(int(patch.n_sources), "sources", launch, mode, flush=True)
                for a, b in zip(*routes(patch, prop, launch, mode)):
                    assert np.all(np.isfinite(a)) and np.array_equal(a, b), (launch, mode)


@pytest.mark.parametrize("n_psf,cap", [(8, MASK_CAP), (57, ACT_CAP)])
def test_more_gaussians_than_the_lds_tables_hold(hip, n_psf, cap):
    """9216 and 65664 Gaussians an exposure: past the tables every slot of a
    Gaussian, and every Gaussian, is evaluated."""
    side = 48 if cap == MASK_CAP else 16
    spec = PatchSpec(n_sources=128, n_bands=1, n_exp_per_band=1, side=side, n_psf=n_psf)
    patch, prop = make(spec, 10 + n_psf)
    try:
        assert 128 * int(patch.n_psf_per_source[0]) > cap
        if cap == MASK_CAP:
            c_ref, d_ref = oracle.evaluate(patch, prop)
        for K in (1, 8):
            for W in (1, 4):
                for persistent in (0, 1):
                    launch = dict(pix_per_lane=K, waves_per_group=W, persistent=persistent)
                    print(n_psf, launch, flush=True)
                    two, one = routes(patch, prop, launch, "mixed")
                    for a, b in zip(two, one):
                        assert np.all(np.isfinite(a)) and np.array_equal(a, b), launch
                    if cap == MASK_CAP:
                        assert chi2_relerr(one[0], c_ref).max() <= CHI2_RTOL
                        assert not grad_mismatch(one[1], d_ref).any()
    finally:
        patch.free()
