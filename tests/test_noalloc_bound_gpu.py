"""The largest grids that the allocation-free step takes: its bound counts a fixed
size for the control block, so that the same grids are taken and refused however
that grows. 3D MHD: 3328 B + 256 B + 120 B a cell, up to 256, in 128 MiB: 1 118 451
cells."""

import ctypes

import numpy as np
import pytest

from astronomix_amd import _native
from astronomix_amd import workloads as W
from astronomix_amd._finite_volume import native_config
from astronomix_amd.option_classes.simulation_config import HLL

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,taken", [((61, 95, 193), True), ((15, 173, 431), True), ((4, 502, 557), False)])
def test_grids_at_the_bound(gpu, shape, taken):
    import torch
    print(f"[gpu] noalloc bound {shape}", flush=True)
    assert (np.prod(shape) <= 1118451) == taken
    lib = _native.load_library()
    nc = native_config((8,) + shape, W.fv_config(3, shape[-1], mhd=True, riemann=HLL), 5 / 3, 0.3, 1.0 / shape[-1])
    a = torch.from_numpy(W.random_smooth(shape, True, seed=5)).cuda()
    b, dt = a.clone(), torch.empty((), device="cuda")
    ctx = _native.FvContext(_native.AmxFvConfig.from_buffer_copy(nc))
    ctx.cfl_dt(a, dt)
    ctx.evolve_state(a, dt)
    status = lib.amx_fv_evolve_state_noalloc(ctypes.byref(nc), ctypes.c_void_p(b.data_ptr()),
                                             ctypes.c_void_p(dt.data_ptr()), None, None)
    torch.cuda.synchronize()
    if taken:
        assert status == _native.AMX_OK and torch.equal(a, b)
    else:
        assert status != _native.AMX_OK and b"scratch" in lib.amx_last_error()
