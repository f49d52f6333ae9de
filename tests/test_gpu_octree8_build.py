"""The dense octree's builder at the edges of its launches: one, two, three and
four kernels of three levels, cells with no point, with one, with more than a
thread sums and with more codes than are staged."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _points(kind, n, seed):
    rng = np.random.default_rng(seed)
    p = rng.random((n, 3))
    if kind == "heap":  # most points in a few cells, the others anywhere
        k = n - n // 8
        p[:k] = 0.3 + 0.01 * rng.integers(0, 3, (k, 1)) + 1e-5 * p[:k]
    m = rng.uniform(0.5, 1.5, n)
    m[::7] = 0.0
    nrm = rng.normal(size=(n, 3))
    return p.astype(np.float32), nrm.astype(np.float32), m.astype(np.float32)


@pytest.mark.parametrize("kind,n,depth", [
    ("any", 1, 1), ("any", 17, 1), ("heap", 40000, 1), ("heap", 129, 2), ("any", 5000, 3),
    ("heap", 17 * 8, 4), ("heap", 60001, 4), ("any", 2049, 5), ("any", 30000, 6),
    ("heap", 30000, 7), ("any", 1, 8),
])
def test_records_match_the_oracle(gpu, kind, n, depth):
    from sbh_amd import ffi

    p, nrm, m = _points(kind, n, 100 * depth + n)
    lo, hi = np.zeros(3, np.float32), np.ones(3, np.float32)
    args = [torch.tensor(a, device="cuda") for a in (p, nrm, m, lo, hi)]
    leaf, node, contrib = (t.cpu().numpy() for t in
                           ffi.build_octree8_buffers_with_contrib(*args, max_depth=depth))
    rleaf, rnode, rcontrib = O.build_octree8(p, nrm, m, lo, hi, depth)
    np.testing.assert_array_equal(leaf.ravel(), np.asarray(rleaf).view(np.uint8).ravel())
    got = node.reshape(-1, 104)
    want = np.asarray(rnode).view(np.uint8).reshape(-1, 104)
    # everything before the contribution (structure and geometry) to the byte
    np.testing.assert_array_equal(got[:, :72], want[:, :72])
    # the contributions against sums in 64 bits: a leaf of c points rounds at most c
    # times, a parent 8 times a level, the quotient and products a few more
    g, w = got[:, 72:].copy().view(np.float32), want[:, 72:].copy().view(np.float32)
    count = (want[:, 4:8].copy().view(np.uint32) - want[:, 0:4].copy().view(np.uint32)).max()
    eps = (count + 8 * depth + 4) * 2.0 ** -24
    np.testing.assert_allclose(g, w, rtol=0, atol=eps * max(1.0, np.abs(w).max()))
    np.testing.assert_array_equal(contrib.ravel(), got[:, 72:].ravel())
