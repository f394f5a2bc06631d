"""The size defaults' passes (tiles held in registers, tiles pipelined over a workgroup's waves)
against the CPU oracle, bit for bit, at the edges of their strips and tiles."""
import numpy as np
import pytest
import torch

import sfhip
from oracle import sf_oracle as O

import cases

pytestmark = pytest.mark.gpu

STATE = ("P", "Vx_s", "Vy_s", "dVx", "dVy")


def _compare(S, nx, ny, n_iter):
    args = (1.3, 0.9 / (nx - 1), 1.1 / (ny - 1))
    G = {k: sfhip.from_numpy(S[k]) for k in STATE + ("rho_vy", "mu_b", "mu_p")}
    sfhip.set_pt_fusion(nx, ny, 0, 0)
    sfhip.pt_iterations(n_iter, G["P"], G["Vx_s"], G["Vy_s"], G["dVx"], G["dVy"], G["rho_vy"], G["mu_b"], G["mu_p"],
                        *args, nx, ny, 0.01)
    torch.cuda.synchronize()
    O.compute_timesteps(S, nx, ny, *args[1:])
    O.pt_iterations(S, nx, ny, n_iter, *args, 0.01)
    for k in STATE:
        assert np.array_equal(sfhip.to_numpy(G[k]), S[k], equal_nan=True), (nx, ny, n_iter, k)


# grids of one strip and one tile, one column or row past it, several rows per wave, and (from 745
# nodes per side) the pipelined pass with tiles that end on, before and after the last row
@pytest.mark.parametrize("nx,ny", [(3, 3), (4, 17), (50, 4), (51, 5), (52, 9), (101, 64), (103, 131), (301, 257), (450, 449),
                                   (640, 333), (760, 745), (801, 800), (1001, 777), (2301, 401)])
def test_size_default_passes_bitwise(gpu, nx, ny):
    n_iter = 2 * 7 + 6 + 1 if nx >= 700 else 41  # whole passes and a remainder
    _compare(cases.random_state(nx, ny, seed=nx * 13 + ny), nx, ny, n_iter)


@pytest.mark.parametrize("nx,ny", [(70, 40), (770, 760)])
@pytest.mark.parametrize("log2_mu", [-260, 260])
def test_size_default_passes_extreme_viscosity(gpu, nx, ny, log2_mu):
    """Rows whose viscosity leaves the range of the short division sequence take the full one (the
    scheme overflows with 2^-260: infinities and NaN then stand where the oracle has them)."""
    S = cases.random_state(nx, ny, seed=5)
    S["mu_p"][:, ny // 3: ny // 2] *= 2.0 ** log2_mu
    for k in STATE:
        S[k][:] = 0.0
    _compare(S, nx, ny, 15)


def test_pipelined_pass_4096_bitwise(gpu):
    """The kernel of 4096^2 solves at that size: two pipelined passes of seven iterations and one of four
    (a run of less than two whole passes keeps the one-wave ones)."""
    n = 4096
    sfhip.time_passes(n, n, True)
    try:
        _compare(cases.random_state(n, n, seed=4097, scale=1e-3, contrast=4.0), n, n, 18)
        launches = sfhip.pass_times(n, n)
    finally:
        sfhip.time_passes(n, n, False)
    assert sorted((t["precision"], t["iters_per_launch"], t["launches"]) for t in launches) == [(0, 4, 1), (0, 7, 2)]


def test_flat_grid_bitwise(gpu):
    """A flat grid of 1,786 strips keeps the one-wave passes of four iterations."""
    nx, ny = 100000, 5
    sfhip.time_passes(nx, ny, True)
    try:
        _compare(cases.random_state(nx, ny, seed=11), nx, ny, 19)
        launches = sfhip.pass_times(nx, ny)
    finally:
        sfhip.time_passes(nx, ny, False)
    assert sorted((t["iters_per_launch"], t["launches"]) for t in launches) == [(3, 1), (4, 4)]


@pytest.mark.parametrize("n_iter,passes", [(2, {}), (3, {2: 1}), (4, {2: 2}), (7, {3: 1, 4: 1}), (14, {7: 2}),
                                           (15, {3: 1, 4: 3}), (21, {5: 3, 6: 1}), (28, {7: 4})])
def test_resident_runs_end_in_the_callers_arrays(gpu, n_iter, passes):
    """Runs of resident passes take an even number of launches (single iterations are not timed), so
    nothing is copied back."""
    nx, ny = 64, 64
    sfhip.time_passes(nx, ny, True)
    try:
        _compare(cases.random_state(nx, ny, seed=n_iter), nx, ny, n_iter)
        launches = {t["iters_per_launch"]: t["launches"] for t in sfhip.pass_times(nx, ny)}
    finally:
        sfhip.time_passes(nx, ny, False)
    assert launches == passes
