"""Attenuated direct sums over many sources: each query's terms go to one running
sum in the order of the sources, rounding for rounding."""
import numpy as np
import pytest
from scipy.special import erfc

pytestmark = pytest.mark.gpu

EPS, RC = 0.05, 2.0


def _terms(q, g, p, m):
    """Terms of the force and of the query-side VJP at one query in 64 bits."""
    d = q.astype(np.float64) - p.astype(np.float64)
    r2 = (d * d).sum(1)
    s = (r2 + EPS * EPS + 1e-12) ** -0.5
    r = np.sqrt(r2 + 1e-12)
    u = r / (2.0 * RC)
    e = np.exp(-u * u)
    lin = s ** 3 * (erfc(u) + 2.0 / np.sqrt(np.pi) * u * e)
    k = (d @ g) * (3.0 * lin * s * s + s ** 3 * r * e / (2.0 * np.sqrt(np.pi) * RC ** 3))
    return -(m * lin)[:, None] * d, -m[:, None] * (lin[:, None] * g - k[:, None] * d)


# either side of the line, and of the one between 16 and 4 lanes per query; ends
# of the source tiles (64 and 16 a time) and of the query blocks
@pytest.mark.parametrize("n,m", [(65536, 1), (65536, 17), (65551, 16383), (65537, 16385),
                                 (65535, 17)])
def test_sums_in_source_order(gpu, n, m):
    from sbh_amd import ffi

    rng = np.random.default_rng(n)
    p = rng.uniform(0.0, 1.0, (n, 3)).astype(np.float32)
    # the first source heavy, the others each below half an ulp of its term
    p[0] = 0.9
    w = np.full(n, 1e-9, np.float32)
    w[0] = 1.0
    q = rng.uniform(-0.6, -0.4, (m, 3)).astype(np.float32)
    g = rng.uniform(0.5, 1.0, (m, 3)).astype(np.float32)
    kw = dict(softening_scale=EPS, cutoff_scale=RC)
    out = [ffi.softened_direct_force(p, w, q, **kw).cpu().numpy(),
           ffi.softened_direct_force_vjp(p, w, q, g, **kw).cpu().numpy()]
    rows = np.unique(np.r_[0:min(m, 20), max(0, m - 20):m])
    whole, running = [[], []], [[], []]
    for r in rows:
        for k, t in enumerate(_terms(q[r], g[r].astype(np.float64), p, w.astype(np.float64))):
            whole[k].append(t.sum(0))
            running[k].append(np.add.accumulate(t.astype(np.float32), 0, dtype=np.float32)[-1])
    rel = lambda a, b: np.linalg.norm(a - b) / np.linalg.norm(b)
    for k in range(2):
        a, ref = np.array(whole[k]), np.array(running[k], np.float64)
        lost = rel(ref, a)
        assert lost > 2e-5  # of the light sources, which the running sum loses
        if n < 65536:
            assert rel(out[k][rows], a) < 0.5 * lost  # split sums keep most of them
        else:
            # the one term that counts: about 10 roundings of 6e-8
            assert rel(out[k][rows], ref) < 6e-7
            few = [ffi.softened_direct_force(p, w, q[:5], **kw),
                   ffi.softened_direct_force_vjp(p, w, q[:5], g[:5], **kw)][k]
            np.testing.assert_array_equal(few.cpu().numpy(), out[k][:5])
