"""Adjoints of 3,000,000 points and more in all run by single waves: the same
gradients as from the sets alone, which teams of waves walk, and as the oracle's."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", [1, 2, 3])
def test_large_forest_adjoint_matches_its_sets(gpu, order):
    from sbh_amd import gravity as G

    sizes = [620011, 1, 65, 690000, 1690000]
    n = sum(sizes)
    assert n >= 3000000
    g = torch.Generator(device="cuda").manual_seed(order)
    p = torch.rand((n, 3), generator=g, device="cuda")
    m = torch.rand(n, generator=g, device="cuda") / n
    c = torch.randn((n, 3), generator=g, device="cuda")
    kw = dict(softening_scale=0.01, leaf_size=32, multipole_order=order)
    gx, gm = G.gravity_force_vjp_batch(p, m, c, G.set_offsets(sizes, device="cuda"), **kw)
    lo = 0
    for k in sizes:
        s = slice(lo, lo + k)
        lo += k
        if k < 2:
            continue
        rx, rm = G.gravity_force_vjp(p[s].contiguous(), m[s].contiguous(), c[s].contiguous(), **kw)
        for a, r in ((gx[s], rx), (gm[s], rm)):
            # sums of up to 1e4 terms in another order, partly by atomics: some 1e-6
            err = ((a - r).double().norm() / r.double().norm()).item()
            assert np.isfinite(err) and err < 1e-5


@pytest.mark.parametrize("order", [1, 2, 3])
def test_sets_of_a_large_call_match_oracle(gpu, order):
    from sbh_amd import gravity as G

    # the walk is chosen by the points in all; two small sets are checked
    sizes = [5003, 2990000, 6000]
    n = sum(sizes)
    assert n >= 3000000
    g = torch.Generator(device="cuda").manual_seed(7 + order)
    p = torch.rand((n, 3), generator=g, device="cuda")
    m = torch.rand(n, generator=g, device="cuda") / n
    c = torch.randn((n, 3), generator=g, device="cuda")
    eps = 0.02
    gx, gm = G.gravity_force_vjp_batch(p, m, c, G.set_offsets(sizes, device="cuda"),
                                       softening_scale=eps, leaf_size=16, multipole_order=order)
    for s in (slice(0, 5003), slice(n - 6000, n)):
        P, M, C, X, W = (t[s].cpu().numpy() for t in (p, m, c, gx, gm))
        T = O.Tree(P, M, max_depth=10, leaf_size=16)
        r = T.eval(beta=2.0, eps=eps, use_quad={1: 0, 2: 1, 3: 2}[order], cot_sorted=C[T.perm])
        # sums of thousands of terms of about 10 roundings each
        assert O.rel_l2(X[T.perm], r["gq"] + r["gsx"]) < 1e-5
        assert O.rel_l2(W[T.perm], r["gsm"]) < 1e-5
