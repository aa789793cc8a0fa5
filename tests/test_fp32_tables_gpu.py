"""The anchor-block tables of the FP32 pair stage at the edges of their blocks
of 64 poses: the adjacency equals the FP64 path's bit for bit and the distances
agree to FP32 rounding; the adjacency also where the first pose lies far from
the origin."""
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


def _graph(n, seed):
    g = synth.se3_helix(n_poses=300, n_lc=90, outlier_frac=0.3, seed=seed)
    rng = np.random.default_rng(seed)
    # keep the first n poses; loop closures end where they can, some at the
    # block edges
    frm = rng.integers(0, n, 90).astype(np.int32)
    to = rng.integers(0, n, 90).astype(np.int32)
    edges = [k for k in (0, 1, 62, 63, 64, 65, 127, 128, n - 1) if k < n]
    frm[: len(edges)] = edges
    to = np.where(to == frm, (to + 1) % n, to).astype(np.int32)
    # relative poses of the folded trajectory, translations a little off
    tr = O.fold(3, g.pose0, g.odom[: n - 1], g.odom_cov[: n - 1])
    R, t = tr[:, :9].reshape(-1, 3, 3), tr[:, 9:12]
    Rr = R[frm].transpose(0, 2, 1) @ R[to]
    tt = np.einsum("kji,kj->ki", R[frm], t[to] - t[frm]) + 0.05 * rng.standard_normal((90, 3))
    T = np.concatenate([Rr.reshape(-1, 9), tt], axis=1)
    return g, g.odom[: n - 1], g.odom_cov[: n - 1], frm, to, T, g.lc_cov[:90]


@pytest.mark.parametrize("special", ["plain", "far"])
@pytest.mark.parametrize("n", [2, 63, 64, 65, 127, 128, 129, 193])
def test_block_edges(ctx, n, special):
    g, odom, cov, frm, to, T, C = _graph(n, 7 * n)
    pose0 = np.array(g.pose0, dtype=np.float64)
    if special == "far":
        pose0.reshape(-1)[9:12] += 1e6
    print(f"[fp32 tables] n={n} {special}", flush=True)
    ctx.pcm_upload(3, pose0, odom, cov, frm, to, T, C)
    ctx.pcm_run(-1.0, 5.0, precision=_capi.PCM_FP64_REPLAY, want_dist=True)
    ref = ctx.pcm_download(want_dist=True)
    ctx.pcm_run(-1.0, 5.0, precision=_capi.PCM_FP32_RECHECK, want_dist=True)
    got = ctx.pcm_download(want_dist=True)
    assert np.array_equal(got["adj_bits"], ref["adj_bits"])
    if special == "plain":
        # the bound the recheck band stands on
        m = len(ref["accepted"])
        iu = np.triu_indices(m, 1)
        d, r = got["dist"][iu], ref["dist"][iu]
        fin = np.isfinite(r) & (r > 0) & (r < 1e6)
        assert not fin.any() or np.max(np.abs(d[fin] - r[fin]) / r[fin]) < 1e-3
