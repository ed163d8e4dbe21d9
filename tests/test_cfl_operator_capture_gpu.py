"""The CFL operator after a step loop on the same context, captured into a graph
and replayed: its dt depends on the state alone, whatever the loop left behind."""

import pytest

from astronomix_amd import _native
from astronomix_amd import workloads as W
from astronomix_amd._finite_volume import native_config
from astronomix_amd.option_classes.simulation_config import HLL

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,mhd", [((40, 70), False), ((40, 70), True), ((12, 14, 16), False), ((12, 14, 16), True)])
def test_operator_depends_on_its_state_alone(gpu, shape, mhd):
    import torch
    print(f"[gpu] cfl capture {shape} mhd={mhd}", flush=True)
    dim = len(shape)
    slow = torch.from_numpy(W.random_smooth(shape, mhd, seed=7)).cuda()
    fast = slow.clone()
    fast[1:dim + 1] += 5.0

    def context():
        cfg = W.fv_config(dim, shape[-1], mhd=mhd, riemann=HLL)
        return _native.FvContext(native_config(slow.shape, cfg, 5 / 3, 0.4, 1.0 / shape[-1]))

    def loop(ctx):
        run = _native.AmxFvRun(t_end=1.0, fixed_timestep=0, num_timesteps=0, exact_end_time=1, max_steps=3)
        ctx.time_integration(fast.clone(), run)

    want, other = torch.empty((), device="cuda"), torch.empty((), device="cuda")
    context().cfl_dt(slow, want)
    context().cfl_dt(fast, other)
    want = want.item()
    assert other.item() < 0.9 * want
    ctx, dt, direct = context(), torch.zeros((), device="cuda"), torch.zeros((), device="cuda")

    def capture():
        g = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(g):
            ctx.cfl_dt(slow, dt)
        return g

    # captured after a loop, then called directly
    loop(ctx)
    behind_loop = capture()
    ctx.cfl_dt(slow, direct)
    assert direct.item() == want
    # captured after the operator, replayed behind a loop
    behind_call = capture()
    for g in (behind_call, behind_loop, behind_call):
        for _ in range(2):
            loop(ctx)
            dt.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert dt.item() == want
        ctx.cfl_dt(fast, direct)
        assert direct.item() == other.item()
