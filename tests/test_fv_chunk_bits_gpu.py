"""A 3D step gives the same bits whatever chunk of planes along x a block of the
stage kernels takes (AMX_LX), for every solver and limiter: the arithmetic of a
cell and of an interface is fused alike before a chunk's first plane, in the
plane loop and behind it."""

import numpy as np
import pytest

from astronomix_amd import _native
from astronomix_amd import workloads as W
from astronomix_amd._finite_volume import native_config
from astronomix_amd.option_classes.simulation_config import (
    AM_HLLC, DOUBLE_MINMOD, HLL, HLLC, HLLC_LM, HYBRID_HLLC, LAX_FRIEDRICHS, MINMOD, OSHER, SUPERBEE, VAN_ALBADA,
    VAN_ALBADA_PP)

pytestmark = pytest.mark.gpu
CASES = [(rs, MINMOD, False) for rs in (HLL, HLLC, HLLC_LM, LAX_FRIEDRICHS, HYBRID_HLLC, AM_HLLC)]
CASES += [(HLL, lim, False) for lim in (OSHER, DOUBLE_MINMOD, SUPERBEE, VAN_ALBADA, VAN_ALBADA_PP)]
CASES += [(HLLC, MINMOD, True), (HLLC, VAN_ALBADA, True)]


@pytest.mark.parametrize("mhd", [False, True])
@pytest.mark.parametrize("riemann,limiter,opened", CASES)
@pytest.mark.parametrize("tiny", [False, True])
def test_bits_do_not_depend_on_the_chunk(gpu, monkeypatch, mhd, riemann, limiter, opened, tiny):
    import torch
    print(f"[gpu] chunks mhd={mhd} rs={riemann} lim={limiter} open={opened} tiny={tiny}", flush=True)
    shape = (33, 20, 70)
    s = W.random_smooth(shape, mhd, seed=3)
    s += 0.02 * np.random.default_rng(3).standard_normal(s.shape).astype(np.float32)
    if tiny:  # subnormal velocities and fields, as ahead of a front
        s[0], s[4] = 1.0, 1.0
        s[1:4] *= 2e-41
        s[5:] *= 2e-41
    cfg = W.fv_config(3, shape[-1], mhd=mhd, riemann=riemann)._replace(limiter=limiter)
    nat = native_config(s.shape, cfg, 5 / 3, 0.4, 1.0 / shape[-1])
    for k in range(6):
        nat.boundary[k] = _native.AMX_BC_OPEN if opened else _native.AMX_BC_PERIODIC
    out = {}
    for lx in (1, 3, 8, 16, 33):
        monkeypatch.setenv("AMX_LX", str(lx))
        ctx = _native.FvContext(_native.AmxFvConfig.from_buffer_copy(nat))
        w, dt = torch.from_numpy(s).cuda(), torch.empty((), device="cuda")
        for _ in range(2):
            ctx.cfl_dt(w, dt)
            ctx.evolve_state(w, dt)
        out[lx] = w
    assert torch.isfinite(out[1]).all()
    for lx in (3, 8, 16, 33):
        assert torch.equal(out[lx], out[1]), lx
