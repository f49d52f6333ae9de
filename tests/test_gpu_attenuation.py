"""The short-range attenuation at cutoffs far from 1: its constants stay finite, so
that pairs far beyond a tiny cutoff contribute 0, and its error stays that of 32 bits."""
import math

import numpy as np
import pytest
import torch
from scipy.special import erfc

pytestmark = pytest.mark.gpu


# 2 sqrt(pi) rc^3 leaves the range of a 32-bit reciprocal below 9e-14
@pytest.mark.parametrize("rc", [2e-15, 1e-14, 9e-14, 1e-10, 1e13])
def test_cutoffs_at_the_ends_of_the_range(gpu, rc):
    from sbh_amd import ffi

    rng = np.random.default_rng(3)
    p = rng.uniform(0, 1, (100, 3)).astype(np.float32)
    m = rng.uniform(0.5, 1.5, 100).astype(np.float32)
    q = rng.uniform(0, 1, (70, 3)).astype(np.float32)
    c = rng.normal(size=(70, 3)).astype(np.float32)
    kw = dict(softening_scale=0.05, cutoff_scale=rc)
    inf = dict(softening_scale=0.05, cutoff_scale=float("inf"))
    leaf, node = ffi.build_octree8_buffers(p, np.zeros_like(p), m, max_depth=3)
    o8 = dict(beta=float("inf"), prune_enabled=False)
    full = ffi.softened_direct_force_full_vjp(p, m, rng.normal(size=(100, 3)).astype(np.float32),
                                              **kw)
    got = [ffi.softened_direct_force(p, m, q, **kw), ffi.softened_direct_force_vjp(p, m, q, c, **kw),
           ffi.softened_barnes_hut_force_octree8(leaf, node, q, **o8, **kw),
           ffi.softened_barnes_hut_force_octree8_vjp(leaf, node, q, c, **o8, **kw), *full]
    want = [ffi.softened_direct_force(p, m, q, **inf),
            ffi.softened_direct_force_vjp(p, m, q, c, **inf)] * 2
    for k, t in enumerate(got):
        assert torch.isfinite(t).all(), k
        if rc < 1:  # every pair lies beyond 1e9 cutoffs (a point's pair with itself is left out)
            assert not t.any(), k
        elif k < 4:  # no pair notices a cutoff of 1e13
            torch.testing.assert_close(t, want[k], rtol=1e-5, atol=1e-5 * float(want[k].abs().max()))


def test_error_of_a_pair_per_range(gpu):
    from sbh_amd import ffi

    rng = np.random.default_rng(0)
    edges = [0, 0.5, 1, 1.5, 2, 3, 4, 6, 8]
    sums = np.zeros((8, 2))
    for rc in (0.05, 0.3, 0.77, 1.0, 1.13, 2.9, 3.3, 30.0):
        r = (rng.uniform(1e-3, 8, 100000) * 2 * rc).astype(np.float32)
        q = np.stack([r, 0 * r, 0 * r], 1)
        f = ffi.softened_direct_force(np.zeros((1, 3), np.float32), np.ones(1, np.float32), q,
                                      softening_scale=0.0, cutoff_scale=rc)
        rd = r.astype(np.float64)
        s2 = rd * rd + 1e-12
        u = np.sqrt(s2) / (2 * np.float64(np.float32(rc)))
        att = erfc(u) + 2 / math.sqrt(math.pi) * u * np.exp(-u * u)
        e = (-f.cpu().numpy()[:, 0] * s2 ** 1.5 / rd / att - 1) ** 2
        k = np.digitize(u, edges) - 1
        for b in range(8):
            sums[b] += e[k == b].sum(), (k == b).sum()
    rms = np.sqrt(sums[:, 0] / sums[:, 1])
    # roundings of 3.4e-8 (root mean square; one in the reciprocal square root, which
    # its cube triples: 3^2), about ten more of the kernel and the fit, and three
    # of u^2, which e^-u^2 multiplies by u^2 <= edge^2
    assert np.all(rms < 3.4e-8 * np.sqrt(9 + 10 + 3 * np.square(edges[1:]) ** 2)), rms
