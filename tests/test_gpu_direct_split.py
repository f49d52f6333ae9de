"""GPU direct sums at the edges of their split over waves and blocks, and the
short-range attenuation they share with the tree walks, against 64 bits."""
import math

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


@pytest.mark.parametrize("rc", [0.05, 1.0, 30.0])
def test_attenuation_of_a_pair(gpu, rc):
    # One unit source and eps = 0: force r^2 = att(u), u = r / (2 rc), times
    # the rounding of r s^3 (reciprocal square root 1 ulp, cubed, and four
    # products: 7 x 1.2e-7 at most).  att itself: exponential, fit and product
    # within 2.5e-7 of 1, and its argument u^2 to 3 roundings (u^2 e^-u^2 <=
    # 0.37, times 1.8e-7).
    r = np.concatenate([np.geomspace(1e-3, 1, 20000), np.linspace(0.5, 12, 20000)]) * 2 * rc
    r = r.astype(np.float32)
    q = np.stack([r, 0 * r, 0 * r], 1)
    f = _np(_ffi().softened_direct_force(np.zeros((1, 3), np.float32), np.ones(1, np.float32), q,
                                         softening_scale=0.0, cutoff_scale=rc))[:, 0]
    rd = r.astype(np.float64)
    u = rd / (2 * np.float64(np.float32(rc)))
    from scipy.special import erfc

    att = erfc(u) + 2 / math.sqrt(math.pi) * u * np.exp(-u * u)
    s2 = rd * rd + 1e-12
    err = np.abs(-f * s2 ** 1.5 / rd - att)
    assert err.max() < 1.2e-6
    assert np.all(err <= 1e-5 * att + 1e-12)  # the tail too, in relative terms


# Edges of the split: queries around a chunk of 64, sources around a run of 8,
# around one source range per wave (64 each) and where the ranges of the last
# block start beyond the sources; one block per chunk up to 1024 sources (512
# attenuated) and from 65,537 queries on, for many sources two up to there.
@pytest.mark.parametrize("n,m", [(1, 1), (7, 63), (8, 64), (9, 65), (255, 128), (257, 1),
                                 (513, 191), (1024, 70), (1025, 70), (2049, 64), (16385, 3),
                                 (300, 131073), (1500, 65536), (1500, 65537), (1500, 131073)])
@pytest.mark.parametrize("rc,periodic", [(np.inf, False), (np.inf, True), (0.3, False),
                                         (0.3, True)])
def test_split_sums_match_oracle(gpu, n, m, rc, periodic):
    ffi = _ffi()
    rng = np.random.default_rng(n + m)
    p = rng.uniform(0, 1, (n, 3)).astype(np.float32)
    w = rng.uniform(0.5, 1.5, n).astype(np.float32)
    q = rng.uniform(0, 1, (m, 3)).astype(np.float32)
    c = rng.normal(size=(m, 3)).astype(np.float32)
    kw = dict(softening_scale=0.05, cutoff_scale=float(rc), periodic=periodic, box_length=1.0)
    f = _np(ffi.softened_direct_force(p, w, q, **kw))
    g = _np(ffi.softened_direct_force_vjp(p, w, q, c, **kw))
    rows = np.unique(np.concatenate([np.arange(min(m, 200)), np.arange(max(0, m - 70), m)]))
    rf = O.direct_force_soft(p, w, q[rows], 0.05, rc, periodic, 1.0)
    rg = O.direct_force_soft_vjp(p, w, q[rows], c[rows], 0.05, rc, periodic, 1.0)
    # sums of n products of about 8 roundings each, their terms partly cancelling
    np.testing.assert_allclose(f[rows], rf, rtol=2e-4, atol=2e-6 * np.abs(rf).max())
    np.testing.assert_allclose(g[rows], rg, rtol=2e-4, atol=2e-6 * np.abs(rg).max())
    # the full adjoint has no queries; among the 1500^2 pairs of the last rows some lie
    # half a box apart to 3e-8, where 32 and 64 bits may pick opposite images
    if m == 1 or n > 4000 or m > 65536:
        return
    cp = rng.normal(size=p.shape).astype(np.float32)
    gx, gm = ffi.softened_direct_force_full_vjp(p, w, cp, **kw)
    rx, rm = O.direct_full_vjp_cut(p, w, cp, 0.05, rc, periodic, 1.0) if np.isfinite(rc) else \
        O.direct_full_vjp(p, w, cp, 0.05, periodic, 1.0)
    if n > 1:
        assert O.rel_l2(_np(gx), rx) < 1e-5 and O.rel_l2(_np(gm), rm) < 1e-5
    else:  # a lone point's pair with itself is left out
        assert not _np(gx).any() and not _np(gm).any()


def test_split_sums_under_capture_and_from_two_threads(gpu):
    # no scratch under capture: one block per chunk, the same sums to rounding;
    # two host threads on one stream share the scratch, one call at a time
    import threading

    from sbh_amd._lib import buf, call, f32, i32, stream_handle
    from sbh_amd.graph import Graph

    ffi = _ffi()
    rng = np.random.default_rng(5)
    p = torch.tensor(rng.uniform(0, 1, (5000, 3)).astype(np.float32), device="cuda")
    w = torch.full((5000,), 1.0 / 5000, device="cuda")
    eager = ffi.softened_direct_force(p, w, p, cutoff_scale=float("inf"))
    out = torch.empty_like(p)
    g = Graph()
    g.capture(lambda: call("sbh_direct_force_soft", stream_handle(), buf(p), buf(w), buf(p),
                           buf(out), f32(1e-2), f32(float("inf")), i32(0), f32(1.0), i32(256)))
    for _ in range(3):
        out.zero_()
        g.replay()
        np.testing.assert_allclose(_np(out), _np(eager), rtol=1e-4,
                                   atol=2e-6 * float(eager.abs().max()))
        assert torch.equal(ffi.softened_direct_force(p, w, p, cutoff_scale=float("inf")), eager)
    g.close()
    q2 = p[:777].contiguous()
    want = ffi.softened_direct_force(p, w, q2, cutoff_scale=float("inf"))
    got = {}

    def work(k, q):
        got[k] = [ffi.softened_direct_force(p, w, q, cutoff_scale=float("inf"))
                  for _ in range(50)]

    ts = [threading.Thread(target=work, args=a) for a in ((0, p), (1, q2))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    torch.cuda.synchronize()
    assert all(torch.equal(x, eager) for x in got[0])
    assert all(torch.equal(x, want) for x in got[1])
