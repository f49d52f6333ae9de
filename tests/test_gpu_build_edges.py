"""The adaptive tree's build at the edges of its launches: tiles of the topology
and the sort, searches inside and beyond the staged window, levels summed by one
block or by many, and bounding boxes of sets that share a tile."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _G():
    from sbh_amd import gravity

    return gravity


def _points(kind, n, seed):
    rng = np.random.default_rng(seed)
    p = rng.random((n, 3))
    if kind == "clumps":
        p = p * 1e-3 + rng.integers(0, 3, (n, 1))
    elif kind == "repeated":
        p = np.floor(p * 5.0)
    return p.astype(np.float32), rng.uniform(0.5, 1.5, n).astype(np.float32)


# sorts by one block, 2 keys a thread to 2048 points, 4 to 4096; then tiles of 1024
# keys to 2^15, 2048 to 2^17, 4096 above; topology tiles of 1024 points in rounds of
# 64 tiles; leaf sizes about the window's 2048; internal nodes per level about 512 (at leaf size 16 reached near 8700 points)
@pytest.mark.parametrize("kind,n,depth,leaf", [
    ("uniform", 1024, 10, 1), ("clumps", 1025, 10, 32), ("repeated", 2048, 10, 8),
    ("clumps", 2049, 5, 8), ("uniform", 4096, 10, 16), ("repeated", 4097, 10, 8),
    ("uniform", 8703, 10, 16), ("uniform", 8721, 10, 16), ("clumps", 32768, 10, 2048),
    ("clumps", 32769, 10, 2049), ("repeated", 65537, 4, 3000), ("uniform", 131072, 9, 32),
    ("clumps", 131073, 10, 24), ("uniform", 530001, 10, 100),
])
def test_tree_at_launch_edges(gpu, kind, n, depth, leaf):
    G = _G()
    p, m = _points(kind, n, n)
    ws = G.new_workspace(n, depth, leaf)
    G.gravity_force(torch.tensor(p, device="cuda"), torch.tensor(m, device="cuda"),
                    max_depth=depth, leaf_size=leaf, workspace=ws)
    tv = G.read_tree(ws, n, depth, leaf)
    T = O.Tree(p, m, max_depth=depth, leaf_size=leaf)
    assert tv.overflow == 0 and tv.num_nodes == T.num_nodes
    for got, want in ((tv.perm, T.perm), (tv.codes, T.codes), (tv.topo[:, 0], T.start),
                      (tv.topo[:, 1], T.count), (tv.topo[:, 2], T.first_child),
                      (tv.topo[:, 3], T.nchild), (tv.parent, T.parent), (tv.geo, T.geo)):
        np.testing.assert_array_equal(got, want)
    # a node's sum of c points (a leaf's, in rows of 16 lanes) or of 8 children
    # rounds at most c / 16 + 5 times, and once more for the product and the
    # quotient; the levels above add at most 5 + 2 each
    mass, com, _ = T.moments()
    leaves = T.count[np.asarray(T.nchild) == 0].max()
    eps = (leaves / 16 + 7 + 7 * depth) * 2.0 ** -24
    np.testing.assert_allclose(tv.mp[:, 3], mass, rtol=eps)
    np.testing.assert_allclose(tv.mp[:, :3], com, rtol=0, atol=2 * eps * np.abs(p).max())


@pytest.mark.parametrize("sizes", [
    [1] * 400, [255, 1, 256, 3, 0, 253, 2, 700, 64, 63, 65], [5, 3000, 0, 1, 40000, 9, 70000, 31],
])
def test_forest_sets_keep_their_own_boxes(gpu, sizes):
    # every set's sums are those of a tree of its own: a box that took a
    # neighbour's point would move its cells.  (Order of the sums aside.)
    G = _G()
    p, m = _points("clumps", sum(sizes), 11)
    p += np.repeat(np.arange(len(sizes)), sizes)[:, None].astype(np.float32)
    tp, tm = torch.tensor(p, device="cuda"), torch.tensor(m, device="cuda")
    offs = G.set_offsets(sizes, device="cuda")
    f = G.gravity_force_batch(tp, tm, offs, softening_scale=0.01).cpu().numpy()
    lo = 0
    for k in sizes:
        if k > 1:
            own = G.gravity_force(tp[lo:lo + k].contiguous(), tm[lo:lo + k].contiguous(),
                                  softening_scale=0.01).cpu().numpy()
            rms = np.sqrt((own ** 2).mean()) + 1e-30
            np.testing.assert_allclose(f[lo:lo + k] / rms, own / rms, rtol=0, atol=2e-5)
        lo += k
