"""The adaptive walks by teams of waves: results independent of the team's size
and of the launch, large leaves, lists that are evaluated more than once, and
forests that hold sets walked by teams and by single waves."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _G():
    from sbh_amd import gravity

    return gravity


def _np(t):
    torch.cuda.synchronize()
    return t.detach().cpu().numpy()


def _points(n, seed, device=True):
    rng = np.random.default_rng(seed)
    p = (rng.normal(size=(n, 3)) * rng.uniform(0.2, 1.0, (n, 1))).astype(np.float32)
    m = rng.uniform(0.5, 1.5, n).astype(np.float32) / n
    c = rng.normal(size=(n, 3)).astype(np.float32)
    return [torch.tensor(a, device="cuda") for a in (p, m, c)] if device else (p, m, c)


# One call below 98,304 points has teams of 16 waves, the forest above it teams
# of 8; a set of 700,000 points is walked by single waves with monopole terms.
@pytest.mark.parametrize("sizes,orders", [([90000, 1, 0, 20000, 64, 65], (1, 2)),
                                          ([700000, 3000, 0, 700001, 129], (1,)),
                                          ([699999, 5], (1, 2))])
def test_forests_equal_single_sets(gpu, sizes, orders):
    G = _G()
    sets = [_points(n, 10 + k) for k, n in enumerate(sizes)]
    P, M, C = (torch.cat([s[i] for s in sets]) for i in range(3))
    offs = G.set_offsets(sizes)
    rows = np.concatenate([[0], np.cumsum(sizes)])
    for order in orders:
        kw = dict(softening_scale=0.005, leaf_size=32, multipole_order=order)
        st, sv = G.new_stats(), G.new_stats()
        f = _np(G.gravity_force_batch(P, M, offs, stats=st, **kw))
        fv = torch.empty_like(P)
        gx, gm = G.gravity_force_vjp_batch(P, M, C, offs, stats=sv, forces_out=fv, **kw)
        np.testing.assert_array_equal(_np(st)[:4], _np(sv)[:4])
        assert _np(st)[5] == 0 and _np(sv)[5] == 0
        total = np.zeros(3, np.int64)
        for k, n in enumerate(sizes):
            if n == 0:
                continue
            s1 = G.new_stats()
            one = _np(G.gravity_force(*sets[k][:2], stats=s1, **kw))
            np.testing.assert_array_equal(f[rows[k]:rows[k + 1]], one, err_msg=f"set {k}")
            x1, m1, f1 = G.gravity_force_vjp(*sets[k], return_forces=True, **kw)
            np.testing.assert_array_equal(_np(fv)[rows[k]:rows[k + 1]], _np(f1))
            # float atomics in arrival order (fp32 rounding of thousands of terms)
            assert n < 3 or O.rel_l2(_np(gx)[rows[k]:rows[k + 1]], _np(x1)) < 1e-5
            assert n < 3 or O.rel_l2(_np(gm)[rows[k]:rows[k + 1]], _np(m1)) < 1e-5
            total += _np(s1)[:3]
        np.testing.assert_array_equal(_np(st)[:3], total)


def _against_oracle(p, m, c, order, leaf, beta):
    G = _G()
    eps = 0.02
    st = G.new_stats()
    gx, gm, f = G.gravity_force_vjp(p, m, c, beta=beta, softening_scale=eps, leaf_size=leaf,
                                    multipole_order=order, stats=st, return_forces=True)
    f2 = G.gravity_force(p, m, beta=beta, softening_scale=eps, leaf_size=leaf,
                         multipole_order=2 if order == 2 else 1)
    T = O.Tree(p, m, max_depth=10, leaf_size=leaf)
    r = T.eval(beta=beta, eps=eps, use_quad={1: 0, 2: 1, 3: 2}[order], cot_sorted=c[T.perm])
    s = G.stats_dict(st)
    assert (s["far"], s["near"], s["groups"]) == (r["far"], r["near"], r["groups"])
    assert s["overflow"] == 0
    # sums of thousands of terms of about 10 roundings each
    assert O.rel_l2(_np(f)[T.perm], r["force"]) < 1e-5
    assert O.rel_l2(_np(f2)[T.perm], r["force"]) < 1e-5
    assert O.rel_l2(_np(gx)[T.perm], r["gq"] + r["gsx"]) < 1e-5
    assert O.rel_l2(_np(gm)[T.perm], r["gsm"]) < 1e-5


@pytest.mark.parametrize("order", [1, 2, 3])
@pytest.mark.parametrize("same,leaf", [(3000, 8), (129, 64), (0, 400)])
def test_large_leaves_are_dealt_to_all_shares(gpu, order, same, leaf):
    # `same` points share a cell down to the depth limit; leaves of up to 400
    p, m, c = _points(6000, 3, device=False)
    p[:same] = p[0] + 1e-5 * np.random.default_rng(0).normal(size=(same, 3)).astype(np.float32)
    _against_oracle(p, m, c, order, leaf, 2.0)


@pytest.mark.parametrize("order", [1, 2, 3])
@pytest.mark.parametrize("n,leaf,beta", [(20000, 2, 2.0), (12000, 1, 6.0), (70001, 16, 3.0)])
def test_lists_evaluated_more_than_once(gpu, order, n, leaf, beta):
    # thousands of accepted nodes and near leaves per group
    _against_oracle(*_points(n, 4, device=False), order, leaf, beta)
