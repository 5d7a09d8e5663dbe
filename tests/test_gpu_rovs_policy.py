"""The policy kernels of the smoothed gradient group a workgroup's paths by
control: the sizes where the grouping changes form (column tiles shared by the
waves, one or two per wave; every control's product above 256 patches with
more than four controls or above 128 with eight; path counts that are no whole
quads or tiles; few paths, which take 8 rows a workgroup or 32 in the form of
every control, and many, which take up to 160), against the FP64 oracle on the
same streams.

Bounds: the FP32 state of T years carries T roundings of at most 2^-23 per
product and growth step and the survival matrices one of 2^-24; the smoothed
validity multiplies a population's relative error by A / tau <= 50 / 4
(tau = 0.02 threshold, sigmoid slope at most 1/4, up to the spread of A around
the threshold): T 2^-22 x 12.5 <= 1.5e-5 at T = 5, as the bound of 2e-5 the
gradient is held to elsewhere."""
import numpy as np
import pytest

from transportoptimiser_amd import rov_species as rs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P,C,N", [
    (32, 8, 37),     # two column tiles, four waves each; eight groups of 8 rows
    (40, 7, 150),    # seven groups at most
    (96, 2, 33),     # four column tiles, two waves each
    (160, 3, 41),    # six column tiles, two idle waves
    (250, 4, 261),   # eight column tiles, a partial one
    (250, 8, 37),    # every control's product
    (257, 3, 70),    # two column tiles for some waves
    (300, 5, 41),    # every control's product, two column tiles
    (512, 4, 45),    # the most patches
    (16, 3, 1),      # one path
])
def test_groups_match_oracle(ctx, oracle, P, C, N):
    pol = np.random.default_rng(P).integers(0, C, size=(4, N)).astype(np.int32)
    pol[1] = C - 1  # a year of one group
    _check(ctx, oracle, P, pol, C)


# Rows of a workgroup in the forward pass and the reverse sweep as the plan
# chooses them on 256 CUs (tests/native/rovs_group_check.cpp holds it to them):
# groups over 32 rows and pairs of row tiles, rows in the second and third
# ballot, dots over several 64-row groups, a last workgroup of few paths.
@pytest.mark.parametrize("P,C,N", [
    (40, 3, 33001),   # 132 and 132
    (40, 8, 39985),   # 160 and 160: twelve group tiles at most
    (100, 7, 20005),  # 80 and 80
    (130, 3, 30011),  # 120 and 60, six column tiles: two idle waves
    (200, 2, 33003),  # 132 and 68
    (257, 2, 10011),  # 40 and 40, two column tiles for some waves
])
def test_many_paths_match_oracle(ctx, oracle, P, C, N):
    pol = np.random.default_rng(P).integers(0, C, size=(3, N)).astype(np.int32)
    pol[1] = 0  # one group of all rows
    pol[2, : N // 2] = C - 1  # workgroups of one group beside mixed ones
    _check(ctx, oracle, P, pol, C)


@pytest.mark.parametrize("P", [48, 200, 300])
def test_eight_controls_most_paths_under_one(ctx, oracle, P):
    # Every control taken in each 32-path tile, seven of them once: eight
    # groups, in the grouped form (48 patches) and every control's product.
    pol = np.full((4, 70), 7, np.int32)
    for t in range(4):
        for p0 in (0, 32):
            pol[t, p0 + np.random.default_rng([P, t, p0]).permutation(32)[:7]] = np.arange(7)
    _check(ctx, oracle, P, pol, 8)


def _check(ctx, oracle, P, pol, C):
    T, N = pol.shape
    pr = rs.synthetic_problem(seed=5, n_patches=P, n_species=1, n_controls=C, n_paths=N,
                              n_years=T, threshold_ratio=0.97)
    tau = 0.02 * pr.species[0].params[3]
    print(f"grouped rows P={P} C={C} N={N}", flush=True)
    val, g = rs.smooth_value_gradient(ctx, pr, pol, tau)
    ref_val, ref_g = oracle.rovs_smooth_grad(pr, pol, tau)
    assert val == pytest.approx(ref_val, rel=2e-5)
    scale = np.abs(ref_g).reshape(C, -1).max(1)
    assert np.all(np.abs(g - ref_g).reshape(C, -1).max(1) <= 2e-5 * scale)
