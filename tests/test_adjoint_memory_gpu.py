"""What a gradient holds between its forward and backward: the inputs of the
steps that were taken, not room for as many as a record may have."""

import pytest

from astronomix_amd import adjoint
from astronomix_amd import workloads as W
from astronomix_amd.option_classes.simulation_params import SimulationParams

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t_end,every", [(0.004, 50), (0.004, 2000), (0.02, 2000)])
def test_recorded_inputs(gpu, t_end, every):
    import torch
    print(f"[gpu] gradient memory t_end={t_end} every={every}", flush=True)
    n = 128
    cfg = W.fv_config(2, n, mhd=False, riemann=1)
    params = SimulationParams(C_cfl=0.4, t_end=t_end, gamma=5 / 3)
    w = torch.from_numpy(W.random_smooth((n, n), False, seed=9)).cuda().requires_grad_(True)

    def held():
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        out = adjoint.rollout(w, cfg, params, checkpoint_every=every)
        torch.cuda.synchronize()
        return (torch.cuda.memory_allocated() - before) / (w.numel() * 4), out

    held()  # the context's own memory
    states, out = held()
    ctx = out.grad_fn
    steps = len(ctx.dts)
    print(states, steps, flush=True)
    assert 3 < steps < 50
    # the result, the step sizes (256 KB: one state of 128^2) and twice the inputs at most
    assert states <= 2 * steps + 4
    (out ** 2).sum().backward()
    assert torch.isfinite(w.grad).all()
