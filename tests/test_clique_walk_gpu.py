"""The heuristic clique at the edges of its walk: vertex counts around one, two
and four words a lane, whole and broken groups of eight picks, the first size
with the step-parallel replay (320) and the last without.  Sizes and working
buffers equal the FP64 oracle's literal scan up to 1,000 vertices, and above
that the allocation-free scan's, whose replay is the sequential one and whose
walks use no derived rows."""
import numpy as np
import pytest
import torch

import oracle as O
from rpgo_amd import _capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = _capi.Context(0)
    yield c
    c.close()


def _adjacency(n, kind):
    """Symmetric 0/1 rows: a large near-complete block among outliers.  The
    block's vertices are contiguous ("runs": whole groups of eight) or every
    third is an outlier ("broken")."""
    i = np.arange(n, dtype=np.int64)
    inl = (i % 3 != 1) if kind == "broken" else (i // 50) % 4 != 1
    out = np.zeros((n, n), np.uint8)
    for r in range(0, n, 512):
        a = i[r:r + 512, None]
        both = inl[r:r + 512, None] & inl[None]
        lo, hi = np.minimum(a, i), np.maximum(a, i)
        h = (lo * 7919 + hi * 104729 + lo * hi) % 997
        out[r:r + 512] = np.where(both, h >= 12, h < 150)
    np.fill_diagonal(out, 0)
    return out


@pytest.mark.parametrize("kind", ["runs", "broken"])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 257, 319, 320, 321, 700, 1000])
def test_small_equals_oracle(ctx, n, kind):
    adj = _adjacency(n, kind)
    k, idx = ctx.max_clique_bits(_capi.pack_bits(adj), n)
    kr, idxr = O.max_clique_heu_dense(adj)
    print(f"[walk] n={n} {kind} clique {k}/{kr}", flush=True)
    assert k == kr and np.array_equal(idx, idxr)


@pytest.mark.parametrize("n", [4095, 4096, 4097, 8192, 8193, 16400])
def test_large_equals_noalloc(ctx, n):
    bits = _capi.pack_bits(_adjacency(n, "runs" if n % 2 else "broken"))
    dev = torch.from_numpy(bits.view(np.int64)).cuda()
    torch.cuda.synchronize()
    k, idx = ctx.max_clique_bits(bits, n)
    kr, idxr = ctx.max_clique_bits_noalloc(dev.data_ptr(), n)
    print(f"[walk] n={n} clique {k}/{kr}", flush=True)
    assert k == kr and np.array_equal(idx, idxr)
