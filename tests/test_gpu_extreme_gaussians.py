"""Both routes of the pixel pass on Gaussians that the shared-block visits of
the two launches are not made for: not finite, far outside the exposure, or so
thin that their cutoff ellipse is ill conditioned.  One wave per tile (the
zero-allocation entry point) visits them by their cutoff box and leaves out a
slot without a pixel inside the cutoff; the two launches have to agree with it
bit for bit, NaN for NaN."""
import ctypes

import numpy as np
import pytest
import torch

from forcepho_amd import _lib, synth
from forcepho_amd.limits import source_struct_dtype
from forcepho_amd.synth import PatchSpec
from helpers import oracle_render

pytestmark = pytest.mark.gpu

NAN, INF = float("nan"), float("inf")


def _far(prop):
    prop["ra"][1] += 1e18          # finite in pixels, its square is not


def _set(name, value):
    def change(prop):
        prop[name][1] = value
    return change


def _amplitude_overflow(prop):
    prop["fluxes"][1] = 3e38       # finite; times G beyond the largest float


def _thin(q):
    def change(prop):
        prop["q"][1], prop["pa"][1] = q, 0.7
        prop["fluxes"][1] *= 100.0
    return change


EXTREMES = {"far": _far, "nan_ra": _set("ra", NAN), "inf_dec": _set("dec", INF),
            "inf_flux": _set("fluxes", INF), "nan_flux": _set("fluxes", NAN),
            "nan_q": _set("q", NAN), "amplitude": _amplitude_overflow,
            "thin_0.03": _thin(0.03), "thin_1e-3": _thin(1e-3), "thin_1e-5": _thin(1e-5),
            "thin_1e-9": _thin(1e-9)}


@pytest.fixture(scope="module")
def patch(hip):
    spec = PatchSpec(n_sources=4, n_bands=1, n_exp_per_band=2, side=90, n_psf=3,
                     psf_elliptical=True, psf_per_exposure=True)
    p, scene, _ = synth.make_patch(spec, config=62, patch_id=0, return_residual=True,
                                   render=oracle_render)
    p.G = np.full(2, 2.0, dtype=np.float32)
    p.send_to_device()
    yield p, scene
    p.free()


def _both(patch, prop):
    """chi2, dchi2 and residual of the two launches and of one wave per tile."""
    prop_dev = torch.from_numpy(np.ascontiguousarray(prop, dtype=source_struct_dtype)
                                .view(np.uint8).copy()).cuda()
    stream = ctypes.c_void_p(int(torch.cuda.current_stream().cuda_stream))
    lib, out = _lib.lib(), []
    for fn in (lib.fpho_evaluate_async, lib.fpho_evaluate_async_noalloc):
        chi2 = torch.full((1,), 7.0, dtype=torch.float64, device="cuda")
        dchi2 = torch.full((4 * 7,), 7.0, dtype=torch.float64, device="cuda")
        _lib.check(fn(patch.device_patch, _lib.dptr(prop_dev), _lib.dptr(chi2),
                      _lib.dptr(dchi2), stream))
        torch.cuda.synchronize()
        out.append((chi2.cpu().numpy(), dchi2.cpu().numpy().reshape(4, 7),
                    patch.retrieve_array("residual")))
    return out


@pytest.mark.parametrize("name", sorted(EXTREMES))
def test_routes_agree_on_extreme_gaussians(patch, name):
    p, scene = patch
    prop = np.array(scene.get_proposal(), dtype=source_struct_dtype)
    EXTREMES[name](prop)
    wrong = []
    for K in (1, 4, 8):
        for cull in (1, 0):
            p.set_launch(pix_per_lane=K, waves_per_group=2, persistent=0, cull=cull)
            for mode in ("mixed", "mixed_centre", "fp64_reduce"):
                p.set_precision(mode)
                print(name, "K", K, "cull", cull, mode, flush=True)
                two, one = _both(p, prop)
                if not all(np.array_equal(a, b, equal_nan=True) for a, b in zip(two, one)):
                    wrong.append((K, cull, mode, two[0], one[0]))
    assert not wrong, wrong
