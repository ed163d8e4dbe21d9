"""The one-launch reverse of a 2D stage (k_adj_tile) at the edges of its 4 x 64
tiles, and the recorded step loop that the reverse sweep starts from.

The tile kernel and the separate passes with dual-number Jacobians
(AMX_ADJ_DUAL=1) differ only by rounding: the bar is that of the existing
comparison of the two, 2e-5 of the largest entry. The recorded loop makes the
plain loop's kernels on the plain loop's values: equal bits.
"""

import numpy as np
import pytest

from astronomix_amd import _native
from astronomix_amd import workloads as W
from astronomix_amd._finite_volume import native_config

pytestmark = pytest.mark.gpu


def state_of(shape, mhd, seed):
    s = W.random_smooth(shape, mhd, seed=seed, dtype=np.float64)
    return (s + 1e-3 * np.random.default_rng(seed).standard_normal(s.shape)).astype(np.float32)


def context(shape, mhd, riemann):
    cfg = W.fv_config(2, shape[0], mhd=mhd, riemann=riemann)
    return _native.FvContext(native_config((7 if mhd else 4,) + shape, cfg, 5 / 3, 0.4, 1.0 / max(shape)))


# one tile and less, a tile and one more row / column, odd remainders, rows
# that wrap inside a tile's halo
@pytest.mark.parametrize("shape", [(4, 64), (5, 65), (3, 5), (6, 63), (9, 130), (33, 67)])
@pytest.mark.parametrize("riemann", [0, 1])
def test_tile_reverse_equals_separate_passes(gpu, shape, riemann, monkeypatch):
    import torch
    print(f"[gpu] adjoint tile {shape} rs={riemann}", flush=True)
    s = torch.from_numpy(state_of(shape, False, 5)).cuda()
    lam = torch.from_numpy(np.random.default_rng(6).standard_normal(s.shape).astype(np.float32)).cuda()
    ctx = context(shape, False, riemann)
    dt = torch.tensor(0.1 / max(shape), device="cuda")
    out = []
    for duals in ("0", "1"):
        monkeypatch.setenv("AMX_ADJ_DUAL", duals)
        res = torch.empty_like(lam)
        ctx.adjoint_step(s, dt, lam, res)
        torch.cuda.synchronize()
        out.append(res.double())
    assert torch.isfinite(out[0]).all()
    assert (out[0] - out[1]).abs().max() <= 2e-5 * out[1].abs().max()


@pytest.mark.parametrize("mhd", [False, True])
@pytest.mark.parametrize("kept", [0, 3, 40])
def test_recorded_loop_equals_plain_loop_and_single_steps(gpu, mhd, kept):
    import torch
    print(f"[gpu] recorded loop mhd={mhd} kept={kept}", flush=True)
    shape = (40, 36)
    s = state_of(shape, mhd, 8)
    run = _native.AmxFvRun(t_end=0.08, fixed_timestep=0, num_timesteps=0, exact_end_time=1, max_steps=-1)
    plain = torch.from_numpy(s).cuda()
    steps = context(shape, mhd, 0).time_integration(plain, run).steps
    ctx = context(shape, mhd, 0)
    rec = torch.from_numpy(s).cuda()
    inputs = torch.zeros((kept,) + rec.shape, device="cuda")
    dts = torch.zeros(64, device="cuda")
    st = ctx.time_integration_recorded(rec, run, inputs, dts)
    assert st.steps == steps and 3 < steps < 40
    assert torch.equal(rec, plain)
    one = torch.from_numpy(s).cuda()
    for k in range(steps):
        if k < kept:
            assert torch.equal(inputs[k], one), k
        ctx.evolve_state(one, dts[k])
    assert torch.equal(one, plain)
    assert not dts[steps:].any()


def test_gradient_with_and_without_the_record(gpu, monkeypatch):
    """A run that does not fit the record is reversed from its checkpoints: the same gradient."""
    import torch
    from astronomix_amd import adjoint
    from astronomix_amd.option_classes.simulation_params import SimulationParams
    print("[gpu] gradient with and without the record", flush=True)
    s = state_of((36, 36), True, 9)
    cfg = W.fv_config(2, 36, mhd=True, riemann=1)
    params = SimulationParams(C_cfl=0.4, t_end=0.04, gamma=5 / 3)
    grads = []
    for limit in (1 << 30, 0):
        monkeypatch.setattr(adjoint, "RECORD_BYTES", limit)
        w = torch.from_numpy(s).cuda().requires_grad_(True)
        (adjoint.rollout(w, cfg, params, checkpoint_every=3)[0] ** 2).sum().backward()
        w50 = torch.from_numpy(s).cuda().requires_grad_(True)
        (adjoint.rollout(w50, cfg, params, checkpoint_every=50)[0] ** 2).sum().backward()
        grads += [w.grad, w50.grad]
    for g in grads[1:]:
        assert torch.equal(g, grads[0])
