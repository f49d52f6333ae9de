"""Winding number walk by teams of waves: both team sizes about their boundary,
lists that are evaluated more than once, leaves dealt in pieces, few queries."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("freq,m,leaf_size", [
    (6, 1 << 18, 16), (6, (1 << 18) + 1, 16),   # teams of 16 up to 2^18 queries, of 8 above
    (48, 1, 8), (48, 300, 8),                   # thousands of nodes and leaves per group
    (24, 5000, 128), (24, 5000, 300),           # leaves of up to 128 elements, and larger
])
def test_team_walk_matches_oracle(gpu, freq, m, leaf_size):
    from sbh_amd import synthetic as S
    from sbh_amd import wn

    V, F = S.perturbed_sphere(freq, 3)
    c, n, a = S.face_dipoles(V, F)
    q = np.random.default_rng(m).uniform(-1.5, 1.5, (m, 3)).astype(np.float32)
    st = torch.zeros(8, dtype=torch.int64, device="cuda")
    out = wn.winding_number(c, n, a, q, beta=2.0, max_depth=10, leaf_size=leaf_size,
                            stats=st).cpu().numpy()
    T = O.Tree(c, a, max_depth=10, leaf_size=leaf_size)
    ref = T.wn_eval(n, q, beta=2.0)
    s = st.cpu().numpy()
    assert s[5] == 0 and s[3] == T.num_nodes
    assert (s[0], s[1], s[2]) == (ref["far"], ref["near"], ref["groups"])
    # a term is good to 8 ulp (its square root and reciprocal to 1 each) and the
    # largest stands near |n.d| a / d^3 of the nearest element, up to 0.3 here; a
    # share adds at most 1/16 of the terms, in random signs.  (No relative bound: outside
    # the surface terms of both signs cancel, to 1e-4 at the single query.)
    terms = (ref["far"] + ref["near"]) / m
    tol = (8 + np.sqrt(terms / 16 + 16)) * 2.0 ** -24 * max(1.0, np.abs(ref["wn"]).max())
    assert np.abs(out - ref["wn"]).max() < 4 * tol
