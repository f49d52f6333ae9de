"""The octree8 walks' partial sums and wave-wide shortcuts: a query's result may
not depend on how its chunk is shared by waves, on its neighbours, or on which
form of the MAC, prune and minimum image decided for it."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _np(t):
    torch.cuda.synchronize()
    return t.detach().cpu().numpy()


def _ffi():
    from sbh_amd import ffi

    return ffi


def _tree(n, depth, seed, box=2.0):
    rng = np.random.default_rng(seed)
    p = rng.uniform(0, box, (n, 3))
    p[: n // 2] = np.mod(0.1 + 0.05 * rng.normal(size=(n // 2, 3)), box)  # across the corner
    p = np.minimum(p.astype(np.float32), np.float32(box * (1 - 1e-6)))
    m = rng.uniform(0.5, 1.5, n).astype(np.float32)
    leaf, node = _ffi().build_octree8_buffers(p, np.zeros_like(p), m,
                                              min_corner=np.zeros(3, np.float32),
                                              max_corner=np.full(3, box, np.float32),
                                              max_depth=depth)
    return p, leaf, node


# depth 1 and 3: the partial sums divide the root's children, deeper: two
# levels above the leaves
@pytest.mark.parametrize("depth", [1, 3, 4, 6])
@pytest.mark.parametrize("periodic,rc,prune", [(False, np.inf, True), (False, 0.1, True),
                                               (True, 0.1, True), (True, np.inf, False),
                                               (True, 0.3, False)])
def test_walk_of_many_waves_equals_split_walk_and_oracle(gpu, depth, periodic, rc, prune):
    ffi = _ffi()
    p, leaf, node = _tree(4000, depth, depth)
    rng = np.random.default_rng(9)
    # from 262,144 queries on a chunk has one wave, below it four
    q = rng.uniform(-1, 3, (262144 + 65, 3)).astype(np.float32)
    q[:2000] = p[:2000]
    q[2000:2064] += 100.0  # more than 16 boxes away: the general minimum image
    q[3000, 0] = np.nan
    c = rng.normal(size=q.shape).astype(np.float32)
    qt, ct = torch.tensor(q, device="cuda"), torch.tensor(c, device="cuda")
    kw = dict(beta=1.7, softening_scale=0.05, cutoff_scale=float(rc), prune_enabled=prune,
              prune_r_cut_mult=3.0, periodic=periodic, box_length=2.0)
    k = 5000
    for f, kind in ((lambda a, b: ffi.softened_barnes_hut_force_octree8(leaf, node, a, **kw),
                     O.KIND_SOFT),
                    (lambda a, b: ffi.softened_barnes_hut_force_octree8_vjp(leaf, node, a, b,
                                                                            **kw),
                     O.KIND_SOFT_VJP),
                    (lambda a, b: ffi.barnes_hut_force_octree8(leaf, node, a, beta=1.7,
                                                               periodic=periodic,
                                                               box_length=2.0), O.KIND_GRAV)):
        whole = _np(f(qt, ct))
        part = _np(f(qt[:k].contiguous(), ct[:k].contiguous()))
        np.testing.assert_array_equal(whole[:k], part)
        rows = np.r_[0:300, 2000:2064]
        soft = kind != O.KIND_GRAV
        ref, _ = O.bh_octree8(_np(leaf), _np(node), q[rows], kind, 1.7, eps=0.05 if soft else 0.0,
                              rc=rc if soft else 0.0, cot=c[rows], prune_enabled=prune and soft,
                              prune_r_cut_mult=3.0, periodic=periodic, box=2.0)
        # a few thousand terms of about 10 roundings each
        assert O.rel_l2(whole[rows][:300], ref[:300]) < 1e-5
        # far queries: differences of coordinates near 102 round to half of 7.6e-6,
        # 7.6e-5 of the kernel's smallest scale eps = 0.05, times 3 for its cube
        assert O.rel_l2(whole[rows][300:], ref[300:]) < 2.3e-4 or np.abs(ref[300:]).max() < 1e-6


@pytest.mark.parametrize("beta", [0.0, -1.0, 1e-30, 1.5, 1e25, np.inf])
def test_mac_at_the_ends_of_its_range(gpu, beta):
    # beta diameters whose square leaves the fp32 range take the quotient itself
    ffi = _ffi()
    p, leaf, node = _tree(1500, 5, 3)
    q = p[::5].copy()
    out = _np(ffi.softened_barnes_hut_force_octree8(leaf, node, q, beta=beta,
                                                    softening_scale=0.05,
                                                    cutoff_scale=float("inf"),
                                                    prune_enabled=False))
    ref, _ = O.bh_octree8(_np(leaf), _np(node), q, O.KIND_SOFT, beta, eps=0.05, rc=np.inf)
    assert O.rel_l2(out, ref) < 1e-5
