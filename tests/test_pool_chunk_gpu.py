"""A pool's stage launches take the x chunk and the chaining of the span of its
slots: a slot gives the bits of the same simulation alone while the span is wide
and after it has shrunk."""

import numpy as np
import pytest

from astronomix_amd import _native
from astronomix_amd import workloads as W
from astronomix_amd._finite_volume import native_config
from astronomix_amd.option_classes.simulation_config import HLL

pytestmark = pytest.mark.gpu


# 20 slots of the 3D grid make chunks of 12 planes, the slot alone shorter ones;
# one and 20 slots of the 2D grid lie on the two sides of the chaining line
@pytest.mark.parametrize("shape", [(20, 130, 130), (100, 130)])
@pytest.mark.parametrize("batch", [1, 6])
def test_slots_equal_single_runs(gpu, shape, batch):
    import torch
    print(f"[gpu] pool chunks {shape} batch {batch}", flush=True)
    dim = len(shape)
    cfg = native_config((dim + 5,) + shape, W.fv_config(dim, shape[-1], mhd=True, riemann=HLL), 5 / 3, 0.4,
                        1.0 / shape[-1])
    pool = _native.FvPool(cfg, 20)
    pool.set_batch(batch)
    slots = {0: (W.random_smooth(shape, True, seed=1), 0.03), 19: (W.random_smooth(shape, True, seed=2), 0.012)}
    for i, (s, t_end) in slots.items():
        pool.load(i, s, 5 / 3, t_end)
    left = set(slots)
    while left:
        pool.step_launch()
        pool.step_finish()
        for i in sorted(left):
            st = pool.status(i)
            if not st.finished:
                continue
            out = pool.read(i, torch.empty((dim + 5,) + shape, dtype=torch.float32, device="cuda"))
            s, t_end = slots[i]
            alone = torch.from_numpy(s).cuda()
            ctx = _native.FvContext(_native.AmxFvConfig.from_buffer_copy(cfg))
            run = _native.AmxFvRun(t_end=t_end, fixed_timestep=0, num_timesteps=0, exact_end_time=1, max_steps=-1)
            ref = ctx.time_integration(alone, run)
            assert st.steps == ref.steps and 3 < ref.steps and torch.equal(out, alone), i
            pool.release(i)
            left.discard(i)
    pool.close()
