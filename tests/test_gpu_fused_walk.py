"""The adjoint that also returns forces, walked by teams and (monopole terms,
700,000 points and more) by single waves: the values of the separate calls."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# leaf sizes whose ranges end in every remainder of a batch of 8
@pytest.mark.parametrize("n,leaf,order", [(5001, 5, 1), (5001, 7, 3), (100001, 16, 1),
                                          (100001, 13, 3), (40000, 32, 2), (700001, 32, 1),
                                          (700001, 32, 3)])
def test_fused_walk_equals_separate_calls(gpu, n, leaf, order):
    from sbh_amd import gravity as G

    g = torch.Generator(device="cuda").manual_seed(n + leaf)
    p = torch.randn((n, 3), generator=g, device="cuda")
    p[: n // 4] *= 0.05
    m = torch.rand(n, generator=g, device="cuda") / n
    c = torch.randn((n, 3), generator=g, device="cuda")
    kw = dict(softening_scale=0.01, leaf_size=leaf)
    s0, s1 = G.new_stats(), G.new_stats()
    gx, gm, f = G.gravity_force_vjp(p, m, c, multipole_order=order, return_forces=True,
                                    stats=s0, **kw)
    rx, rm = G.gravity_force_vjp(p, m, c, multipole_order=order, stats=s1, **kw)
    rf = G.gravity_force(p, m, multipole_order=2 if order == 2 else 1, **kw)
    assert torch.equal(s0, s1)
    # the same terms, thousands of about 10 roundings each: forces in the same order
    # or (order 3 from 700,000 points on) in another, gradients by atomics in
    # arrival order
    for a, b in ((f, rf), (gx, rx), (gm, rm)):
        assert ((a - b).double().norm() / b.double().norm()).item() < 1e-5
