"""Half pairs of the magnetic fixed point on a GPU: in queued batches of steps
the pair that starts at the previous step's final launch index makes its first
iterate only, and the second one is made where the fixed point goes on. Bits
and iteration counts are those of single steps, which make whole pairs."""

import numpy as np
import pytest

from astronomix_amd import _native
from astronomix_amd import workloads as W
from astronomix_amd._finite_volume import native_config
from astronomix_amd.option_classes.simulation_config import HLL

pytestmark = pytest.mark.gpu


def final_after_even(ks):
    """(previous, next) final launch indices of consecutive steps, previous even and smaller."""
    return {(a, b) for a, b in zip(ks, ks[1:]) if a % 2 == 0 and b > a}


@pytest.mark.parametrize("shape", [(16, 16, 16), (17, 23, 70), (64, 64)], ids=["3d", "3d_odd", "2d"])
def test_loop_calls_of_changing_dt(gpu, shape):
    """Loops of fixed dt on one context drive the final launch index from
    even values up (through the second iterate of a half pair and past it),
    down and back, launch 0 included; each loop equals the same steps alone."""
    import torch
    print(f"[gpu] half pairs, loop calls {shape}", flush=True)
    dim = len(shape)
    state = W.random_smooth(shape, True, seed=8)
    cfg = W.fv_config(dim, shape[-1], mhd=True, riemann=HLL)
    nc = native_config(state.shape, cfg, 5.0 / 3.0, 0.4)
    loop = _native.FvContext(_native.AmxFvConfig.from_buffer_copy(nc))
    single = _native.FvContext(_native.AmxFvConfig.from_buffer_copy(nc))
    s_loop = torch.from_numpy(np.ascontiguousarray(state)).cuda()
    s_step = s_loop.clone()
    ks = []
    for dt, n in [(3e-4, 3), (4e-3, 2), (1e-7, 3), (6e-3, 2), (3e-4, 2), (1e-3, 2), (1e-7, 2), (3e-4, 3), (6e-3, 3)]:
        t_end = float(np.float32(dt) * np.float32(n))
        run = _native.AmxFvRun(t_end=t_end, fixed_timestep=1, num_timesteps=n, exact_end_time=0, max_steps=-1)
        st = loop.time_integration(s_loop, run)
        d = torch.tensor(np.float32(t_end) / np.float32(n), dtype=torch.float32, device="cuda")
        kk = [single.evolve_state(s_step, d) for _ in range(n)]
        torch.cuda.synchronize()
        assert st.steps == n and st.fixed_point_iterations == sum(kk), (dt, st.fixed_point_iterations, kk)
        assert torch.equal(s_loop, s_step), (dt, kk)
        ks += kk
    print(ks, flush=True)
    if shape == (16, 16, 16):
        assert len(final_after_even(ks)) >= 2, ks


@pytest.mark.parametrize("batch", [3, 8])
def test_pool_slots_of_different_counts(gpu, batch):
    """Slots whose final launch indices differ and change share each launch:
    one that its half pair keeps from the rest of the batch goes on from
    there while others are further on or settled."""
    import torch
    print(f"[gpu] half pairs, pool, {batch} steps per launch", flush=True)
    shape = (16, 16, 16)
    cfg = native_config((8,) + shape, W.fv_config(3, 16, mhd=True, riemann=HLL), 5.0 / 3.0, 0.8)
    cfg.fixed_point_tol = 1e-6
    states = [W.random_smooth(shape, True, seed=i, amp=a) for i, a in enumerate((0.05, 0.3, 0.7, 1.0))]
    ends = (0.9, 0.4, 0.2, 0.15)
    alone = []
    for s, te in zip(states, ends):
        ctx = _native.FvContext(_native.AmxFvConfig.from_buffer_copy(cfg))
        w = torch.from_numpy(np.ascontiguousarray(s)).cuda()
        ctx.set_timing(1)  # timed loops take single steps
        run = _native.AmxFvRun(t_end=te, fixed_timestep=0, num_timesteps=0, exact_end_time=1, max_steps=-1)
        st = ctx.time_integration(w, run)
        torch.cuda.synchronize()
        alone.append((w.cpu().numpy(), st))
    means = [st.fixed_point_iterations / st.steps for _, st in alone]
    print(means, [st.steps for _, st in alone], [st.max_fixed_point_iterations for _, st in alone], flush=True)
    assert max(means) - min(means) > 1.0, means
    pool = _native.FvPool(cfg, 4)
    pool.set_batch(batch)
    for i, (s, te) in enumerate(zip(states, ends)):
        pool.load(i, s, 5.0 / 3.0, te)
    status = {}
    while len(status) < 4:
        pool.step_launch()
        pool.step_finish()
        for i in range(4):
            if i not in status and pool.status(i).finished:
                status[i] = pool.status(i)
    for i, (ref, st) in enumerate(alone):
        out = pool.read(i, torch.empty((8,) + shape, dtype=torch.float32, device="cuda")).cpu().numpy()
        assert status[i].steps == st.steps and status[i].fixed_point_iterations == st.fixed_point_iterations, i
        np.testing.assert_array_equal(out, ref)
    pool.close()
