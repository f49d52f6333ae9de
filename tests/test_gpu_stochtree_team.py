"""Stochastic walk with the subdomains of a group dealt to a team's waves: both
team sizes about their boundary, fewer subdomains than shares, one query."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m,leaf", [(3000, 32768, 16), (3000, 32769, 16), (40, 200, 16),
                                      (5, 70, 16), (3000, 1, 8)])
@pytest.mark.parametrize("kind", ["force", "vjp", "wn"])
def test_team_sums_match_oracle(gpu, kind, n, m, leaf):
    from sbh_amd import stochastic as S

    rng = np.random.default_rng(n + m)
    p = rng.normal(size=(n, 3)).astype(np.float32)
    w = (rng.uniform(0.5, 1.5, n) / n).astype(np.float32)
    q = rng.normal(size=(m, 3)).astype(np.float32) * 1.5
    v = rng.normal(size=(max(n, m), 3)).astype(np.float32)
    v /= np.linalg.norm(v, axis=1, keepdims=True)
    st = torch.zeros(8, dtype=torch.int64, device="cuda")
    kw = dict(beta=1.5, samples_per_subdomain=2, seed=5, max_depth=10, leaf_size=leaf, stats=st)
    T = O.Tree(p, w, max_depth=10, leaf_size=leaf)
    ref = dict(beta=1.5, samples=2, seed=5)
    if kind == "force":
        out = S.stochastic_gravity_force(p, w, q, softening_scale=0.05, multipole_order=1, **kw)
        r = T.stoch_eval(q, kind=0, eps=0.05, use_quad=False, **ref)
    elif kind == "vjp":
        out = S.stochastic_gravity_force_vjp(p, w, q, v[:m], softening_scale=0.05,
                                             multipole_order=1, **kw)
        r = T.stoch_eval(q, kind=1, eps=0.05, use_quad=False, cot=v[:m], **ref)
    else:
        out = S.stochastic_winding_number(p, v[:n], w, q, **kw)
        r = T.stoch_eval(q, kind=2, normals=v[:n], **ref)
    s = S.stats_dict(st)
    assert s["overflow"] == 0
    assert (s["node_terms"], s["source_pairs"], s["groups"]) == (r["node"], r["pair"],
                                                                 r["groups"])
    # differences of node and children sums (rounded to about 1e-7 of the node term),
    # weighted by up to n_sub / (P count) of 1e3: 2e-4 of the result's norm
    assert O.rel_l2(out.cpu().numpy(), r["out"]) < 2e-4
