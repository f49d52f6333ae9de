"""The full adjoint of the direct sums leaves a point's pair with itself out: an
infinite or NaN cotangent of a point does not reach its own mass gradient."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [70, 1500])
@pytest.mark.parametrize("rc,periodic", [(np.inf, False), (0.3, False), (0.3, True)])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_own_cotangent_stays_out_of_the_mass_gradient(gpu, n, rc, periodic, bad):
    from sbh_amd import ffi

    rng = np.random.default_rng(n)
    p = rng.uniform(0, 1, (n, 3)).astype(np.float32)
    m = rng.uniform(0.5, 1.5, n).astype(np.float32)
    c = rng.normal(size=(n, 3)).astype(np.float32)
    kw = dict(softening_scale=0.05, cutoff_scale=float(rc), periodic=periodic, box_length=1.0)
    # points at the ends of a wave's chunk and of a run of 8 sources, and in the rest
    for k in (0, 7, 63, 64, n - 1):
        broken = c.copy()
        broken[k] = bad
        gx, gm = (t.cpu().numpy() for t in ffi.softened_direct_force_full_vjp(p, m, broken, **kw))
        zero = c.copy()
        zero[k] = 0.0
        ref = O.direct_full_vjp_cut(p, m, zero, 0.05, rc, periodic, 1.0) if np.isfinite(rc) else \
            O.direct_full_vjp(p, m, zero, 0.05, periodic, 1.0)
        # every other pair of the point is with a finite cotangent
        assert abs(gm[k] - ref[1][k]) < 1e-4 * np.abs(ref[1]).max()
        assert not np.isfinite(np.delete(gm, k)).any() and not np.isfinite(gx[k]).all()
