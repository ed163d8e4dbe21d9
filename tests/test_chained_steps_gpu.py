"""Queued steps that do their control work in their own kernels, against the same
steps taken one at a time with the operators, bit for bit: adaptive dt over
several batches with a clamped last step, both kinds of chain (with and without a
fixed point), one- and two-launch gas steps, and the schemes that do not chain.
A fixed point that needs more launches than were queued (tolerance 1e-7) holds a
chained step, which the host finishes.
"""

import numpy as np
import pytest

from astronomix_amd import _native
from astronomix_amd import workloads as W
from astronomix_amd._finite_volume import native_config
from astronomix_amd.option_classes.simulation_config import HLLC, HLLC_LM, LAX_FRIEDRICHS

pytestmark = pytest.mark.gpu
BIG = (1030, 1027)  # two stage launches a gas step


def context(shape, mhd, riemann, tol):
    dim = len(shape)
    cfg = W.fv_config(dim, shape[-1], mhd=mhd, riemann=riemann)
    nat = native_config(((dim + 2 + (3 if mhd else 0)),) + shape, cfg, 5 / 3, 0.4, 1.0 / shape[-1])
    if tol:
        nat.fixed_point_tol = tol
    return _native.FvContext(nat)


@pytest.mark.parametrize("shape,mhd,riemann,tol", [
    ((40, 70), False, 0, 0), ((40, 70), True, HLLC, 0), (BIG, False, HLLC, 0), (BIG, True, 0, 0),
    ((13, 18, 33), False, HLLC_LM, 0), ((13, 18, 33), True, 0, 0), ((13, 18, 33), True, 0, 1e-7),
    ((40, 70), False, LAX_FRIEDRICHS, 0), ((40, 70), True, LAX_FRIEDRICHS, 0)])
@pytest.mark.parametrize("steps", [1, 4, 5, 23])
def test_loop_equals_operators(gpu, shape, mhd, riemann, tol, steps):
    import torch
    print(f"[gpu] chained {shape} mhd={mhd} rs={riemann} tol={tol} steps={steps}", flush=True)
    s = W.random_smooth(shape, mhd, seed=7)
    ctx = context(shape, mhd, riemann, tol)
    one, dt = torch.from_numpy(s).cuda(), torch.empty((), device="cuda")
    t = np.float32(0)
    for i in range(steps):
        ctx.cfl_dt(one, dt)
        if i == steps - 1:  # the end time cuts the last step short
            t_end = np.float32(t + np.float32(0.6) * np.float32(dt.item()))
            dt.fill_(float(np.float32(t_end - t)))
        ctx.evolve_state(one, dt)
        t = np.float32(t + np.float32(dt.item()))
    run = _native.AmxFvRun(t_end=float(t_end), fixed_timestep=0, num_timesteps=0, exact_end_time=1, max_steps=-1)
    for _ in range(2):  # a second loop on the same context starts from a fresh chain
        out = torch.from_numpy(s).cuda()
        st = ctx.time_integration(out, run)
        assert st.steps == steps and np.float32(st.t) == t
        assert torch.equal(out, one)
