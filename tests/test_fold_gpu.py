"""The odometry fold at the edges of its blocks of 24 steps: trajectory records
bit-equal to the FP64 oracle for every chain length around one, two and three
blocks, with covariances that lack rotation information or hold infinities."""
import numpy as np
import pytest

import oracle as O
from rpgo_amd import _capi, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = _capi.Context(0)
    yield c
    c.close()


def _graph(dim, n, seed):
    if dim == 3:
        return synth.se3_helix(n_poses=max(n, 110), n_lc=2, outlier_frac=1.0, seed=seed)
    return synth.se2_random_walk(n_poses=max(n, 10), n_inlier=2, n_outlier=1, seed=seed)


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("special", ["plain", "no_rotation", "infinite"])
@pytest.mark.parametrize("n", [1, 2, 3, 24, 25, 26, 48, 49, 50, 73])
def test_fold_blocks(ctx, dim, special, n):
    g = _graph(dim, n, 10 * n + dim)
    D = 6 if dim == 3 else 3
    odom = g.odom[: n - 1]
    cov = np.array(g.odom_cov[: n - 1]).reshape(-1, D, D)
    if special == "no_rotation" and n > 2:
        cov[(n - 1) // 2, 0, 0] = np.nan
    if special == "infinite" and n > 2:
        cov[(n - 1) // 2, D - 1, D - 1] = np.inf
    cov = cov.reshape(-1, D * D)
    print(f"[fold] dim={dim} n={n} {special}", flush=True)
    none = np.zeros(0, np.int32)
    ctx.pcm_upload(dim, g.pose0, odom, cov, none, none, g.lc_pose[:0], g.lc_cov[:0])
    ctx.pcm_run(-1.0, 5.0)
    with np.errstate(all="ignore"):
        np.testing.assert_array_equal(ctx.pcm_traj(), O.fold(dim, g.pose0, odom, cov))
