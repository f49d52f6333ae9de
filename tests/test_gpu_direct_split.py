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
