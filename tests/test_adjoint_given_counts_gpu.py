"""The reverse step differentiates as many fixed-point applications as its count
says, whatever was in its workspace: iterates past the settled one are made, not
taken as they lie there."""

import numpy as np
import pytest

from astronomix_amd import _native
from astronomix_amd import workloads as W
from astronomix_amd._finite_volume import native_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(20, 36), (9, 12, 17)])
@pytest.mark.parametrize("more", [0, 1, 2, 5])
def test_count_past_the_settled_iterate(gpu, shape, more):
    import torch
    print(f"[gpu] adjoint count + {more} {shape}", flush=True)
    dim = len(shape)
    cfg = W.fv_config(dim, shape[-1], mhd=True, riemann=1)
    nat = native_config((dim + 5,) + shape, cfg, 5 / 3, 0.4, 1.0 / max(shape))
    a, b = (torch.from_numpy(W.random_smooth(shape, True, seed=i)).cuda() for i in (3, 4))
    lam = torch.from_numpy(np.random.default_rng(6).standard_normal(a.shape).astype(np.float32)).cuda()
    dt = torch.tensor(0.1 / max(shape), device="cuda")
    fresh, used = (_native.FvContext(_native.AmxFvConfig.from_buffer_copy(nat)) for _ in range(2))
    count = fresh.evolve_state(b.clone(), dt)
    # another state's iterates, further than this step's, in the workspace of one
    long = torch.empty_like(lam)
    used.adjoint_step(a, dt, lam, long, count=count + more + 2)
    out, plain = [torch.empty_like(lam) for _ in range(2)], torch.empty_like(lam)
    fresh.adjoint_step(b, dt, lam, out[0], count=count + more)
    used.adjoint_step(b, dt, lam, out[1], count=count + more)
    fresh.adjoint_step(b, dt, lam, plain)
    assert torch.equal(out[0], out[1])
    if more == 0:
        assert torch.equal(out[0], plain)
    # further applications of a map that has settled: the terms they add to the
    # derivative are of the size of its tolerance, 1e-5, times a few tens
    assert (out[0] - plain).abs().max() <= 1e-2 * plain.abs().max()
