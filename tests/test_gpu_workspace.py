"""The workspace of the two-launch pixel pass: when it is asked for, and what
happens where it is not to be had."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

from forcepho_amd import _lib, synth
from forcepho_amd.batch import PatchBatch
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


CHILD = r"""
import ctypes, os, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)   # before the HIP runtime
refuse, refused, count = (ctypes.c_longlong.in_dll(shim, "shim_" + n)
                          for n in ("refuse", "refused", "count"))
sizes = (ctypes.c_longlong * 4096).in_dll(shim, "shim_sizes")
import numpy as np, torch
from forcepho_amd import _lib, synth
from forcepho_amd.limits import source_struct_dtype
from helpers import oracle_render, proposal_for
from test_gpu_workspace import SPEC
_lib.init(0)

def make():
    patch, scene, theta = synth.make_patch(SPEC, config=63, patch_id=0, render=oracle_render)
    patch.send_to_device()
    return patch, np.ascontiguousarray(proposal_for(scene, theta), dtype=source_struct_dtype)

patch, prop = make()
prop_dev = torch.from_numpy(prop.view(np.uint8).copy()).cuda()
chi2 = torch.zeros(2, dtype=torch.float64, device="cuda")
dchi2 = torch.zeros(2 * 5 * 7, dtype=torch.float64, device="cuda")

def stream_ordered(p):
    chi2.zero_(), dchi2.zero_()
    _lib.check(_lib.lib().fpho_evaluate_async(
        p.device_patch, _lib.dptr(prop_dev), _lib.dptr(chi2), _lib.dptr(dchi2),
        ctypes.c_void_p(int(torch.cuda.current_stream().cuda_stream))))
    torch.cuda.synchronize()
    return chi2.cpu().numpy(), dchi2.cpu().numpy().astype(np.float32)

def synchronous(p):
    c, d = p.get_proposer().evaluate_proposal(prop, p)[:2]
    return c, d.reshape(-1)

before = count.value
want = stream_ordered(patch)
asked = list(sizes[before:count.value])
assert len(asked) == 2, asked            # the plan, then its workspace
print("sizes", asked, flush=True)
refuse.value = asked[1]

def five(call, p):
    first = refused.value
    for _ in range(5):
        for a, b in zip(call(p), want):
            assert np.array_equal(a, b)
    return refused.value - first

other, _ = make()
synchronous_tries = five(synchronous, other)
own_tries = five(stream_ordered, other)
other.set_launch()                       # its plan is built anew: asked for once more
rebuilt_tries = five(stream_ordered, other)
patch.free()                             # memory came back: asked for once more
freed_tries = five(synchronous, other)
print("tries", synchronous_tries, own_tries, rebuilt_tries, freed_tries, flush=True)
assert (synchronous_tries, own_tries, rebuilt_tries, freed_tries) == (1, 1, 1, 1)
refuse.value = -1
other.set_launch()
before = count.value
five(stream_ordered, other)
assert asked[1] in sizes[before:count.value]
other.free()
print("done", flush=True)
"""


def test_refused_workspace_is_not_asked_for_on_each_call(hip, tmp_path):
    """Without memory for the workspace a call takes one wave per tile, with the
    same results, and the next call does not try again: a plan asks once, the
    synchronous calls of a device once until a patch is freed."""
    here = os.path.dirname(os.path.abspath(__file__))
    shim = tmp_path / "malloc_shim.so"
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC",
                    os.path.join(here, "native", "malloc_shim.c"), "-o", str(shim), "-ldl"],
                   check=True)
    path = os.pathsep.join([os.path.dirname(here), here, os.environ.get("PYTHONPATH", "")])
    run = subprocess.run([sys.executable, "-u", "-c", CHILD, str(shim)], capture_output=True,
                         text=True, timeout=100, env=dict(os.environ, PYTHONPATH=path))
    print(run.stdout, run.stderr[-3000:], flush=True)
    assert run.returncode == 0 and "done" in run.stdout


def test_freed_and_resent_patches_give_their_memory_back(hip):
    """``free`` of a patch class reaches its device half: sending a patch again
    and freeing it keep no device memory, and a batch keeps the patches it was
    made of until it is freed."""
    spec = PatchSpec(n_sources=1, n_bands=1, n_exp_per_band=4, side=1024, n_psf=1)
    patch, scene, theta = synth.make_patch(spec, config=63, patch_id=1)

    def used():
        torch.cuda.synchronize()
        free, total = torch.cuda.mem_get_info()
        return total - free

    patch.send_to_device()
    prop = proposal_for(scene, theta)
    want = patch.get_proposer().evaluate_proposal(prop, patch)
    one = used()
    pixels = 4 * 4 * spec.npix_unpadded        # bytes of its four pixel arrays
    for _ in range(5):
        patch.send_to_device()
        patch.get_proposer().evaluate_proposal(prop, patch)
    assert used() - one < pixels

    batch = PatchBatch([patch])
    batch.set_proposals([prop])
    patch.free()
    assert patch.device_patch is None
    batch.evaluate()
    torch.cuda.synchronize()
    assert np.array_equal(batch.chi2_host(0), want[0])
    batch.free()
    assert one - used() > pixels
