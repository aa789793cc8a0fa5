"""Appends around the sizes where the route changes: the pinned staging buffer
(32 KB: 85 SE(3) records, a few more keys than records fit) and the one-launch
odometry check (256 loop closures).  Records, accepted loop closures, distances
and adjacency equal a full run's bit for bit, and so do the counts."""
import numpy as np
import pytest

from rpgo_amd import _capi, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctxs():
    c = [_capi.Context(0), _capi.Context(0)]
    yield c
    for k in c:
        k.close()


def _arrays(g, p1, l0, l1):
    return g.lc_from[l0:l1] % p1, g.lc_to[l0:l1] % p1, g.lc_pose[l0:l1], g.lc_cov[l0:l1]


@pytest.mark.parametrize("simple", [False, True])
@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("n_odom,n_lc", [(0, 0), (1, 0), (0, 1), (1, 3), (40, 43), (40, 44), (40, 45), (85, 0), (86, 0),
                                         (0, 255), (0, 256), (0, 257), (300, 300)])
def test_append_sizes(ctxs, dim, simple, n_odom, n_lc):
    g = (synth.se3_helix(n_poses=500, n_lc=330, outlier_frac=0.5, seed=5) if dim == 3 else
         synth.se2_random_walk(n_poses=500, n_inlier=300, n_outlier=30, seed=5))
    thr = (0.1, 0.01, 0.1, 0.01) if simple else (10.0, 5.0)
    run = lambda c: c.pcm_simple_run(*thr) if simple else c.pcm_run(*thr)
    p0, l0 = 120, 20
    p1, l1 = p0 + n_odom, l0 + n_lc
    print(f"[append] dim={dim} simple={simple} +{n_odom} poses +{n_lc} loop closures", flush=True)
    a, b = ctxs
    # loop closures (wrapped into the poses that exist) in two parts
    first, more = _arrays(g, p0, 0, l0), _arrays(g, p1, l0, l1)
    a.pcm_upload(dim, g.pose0, g.odom[: p0 - 1], g.odom_cov[: p0 - 1], *first)
    m0 = run(a).n_accepted
    app = a.pcm_simple_append if simple else a.pcm_append
    sa = app(*thr, odom=g.odom[p0 - 1:p1 - 1], odom_cov=g.odom_cov[p0 - 1:p1 - 1], lc_from=more[0], lc_to=more[1],
             lc_pose=more[2], lc_cov=more[3])
    whole = [np.concatenate([x, y]) for x, y in zip(first, more)]
    b.pcm_upload(dim, g.pose0, g.odom[: p1 - 1], g.odom_cov[: p1 - 1], *whole)
    sb = run(b)
    assert sa.n_accepted == sb.n_accepted >= m0
    da, db = a.pcm_download(), b.pcm_download()
    for k in ("accepted", "odom_dist", "adj_bits"):
        assert np.array_equal(da[k], db[k], equal_nan=k == "odom_dist"), k
    assert np.array_equal(a.pcm_traj(), b.pcm_traj())
    before = np.triu(_capi.unpack_bits(db["adj_bits"], sb.n_accepted), 1)[:m0, :m0].sum() if m0 else 0
    assert sa.n_consistent == sb.n_consistent - before
