"""The WENO kernel's tiles at the sizes where they can go wrong, and its two
forms of the smoothness weights, against the CPU restatement (bar and floor
rule of test_fd_gpu_parity.check_parity)."""

import numpy as np
import pytest

from astronomix_amd.option_classes.simulation_params import SimulationParams
from test_fd_gpu_parity import check_parity, fd, gpu_run, mhd_state, oracle_run  # noqa: F401

pytestmark = pytest.mark.gpu

# (6, 6, 6): the smallest grid; rows shorter than 12 cells take smaller z
# blocks; 101 and 11 end z blocks inside a row; 300 and 520 cut a row into
# blocks; 9 and 17 leave part tiles along x and y.
SHAPES = [(6, 6, 6), (7, 9, 11), (9, 17, 12), (13, 6, 101), (6, 7, 300), (8, 6, 520)]
# velocities in units of the sound speed scaled by k: smoothness indicators
# grow by k^2, so k = 1e5 takes the form with one reciprocal per weight in
# every wave, 1e4 in some, 1 in none
SCALES = [((12, 10, 72), 1e4), ((12, 10, 72), 1e5)]


@pytest.mark.parametrize("shape,k", [(s, 1.0) for s in SHAPES] + SCALES)
def test_weno_tiles_match_oracle(gpu, fd, shape, k):  # noqa: F811
    print(f"[gpu] weno tiles {shape} scale {k:g}", flush=True)
    state = mhd_state(shape, seed=sum(shape))
    state[1:4] *= k
    state[4] *= k * k
    state[5:] *= k
    dt = 0.05 / (max(shape) * k)
    params = SimulationParams(C_cfl=0.4, t_end=2 * dt, dt_max=dt, gamma=5.0 / 3.0)
    kw = dict(fixed=True, num_timesteps=2)
    out, st = gpu_run(state, params, **kw)
    ref, steps, _ = oracle_run(fd, state, params, **kw)
    assert st.steps == steps == 2
    check_parity(fd, f"{shape} x {k:g}", out, ref, state, params, **kw)
