"""The cost-ordered schedule of the walks by single waves (sets of 700,000 points
and more with monopole terms): whatever costs and tags the workspace holds, every
group is walked once."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _G():
    from sbh_amd import gravity

    return gravity


def _points(n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    p = torch.randn((n, 3), generator=g, device="cuda") * torch.rand((n, 1), generator=g,
                                                                     device="cuda")
    m = torch.rand(n, generator=g, device="cuda") / n
    return p, m, torch.randn((n, 3), generator=g, device="cuda")


# one set, and a forest of sets for single waves and for teams
@pytest.mark.parametrize("sizes", [(700000,), (5000, 700001, 64)])
def test_schedule_of_single_waves_changes_no_result(gpu, sizes):
    G = _G()
    n = sum(sizes)
    P, M, C = (torch.cat(t) for t in zip(*(_points(k, k) for k in sizes)))
    offs = G.set_offsets(sizes)
    kw = dict(softening_scale=0.005, max_depth=10, leaf_size=32, multipole_order=1)
    make = lambda: G.new_batch_workspace(n, len(sizes), 10, 32)
    ws = make().zero_()

    def run(ws):
        sf, sv = G.new_stats(), G.new_stats()
        f = G.gravity_force_batch(P, M, offs, workspace=ws, stats=sf, **kw)
        gx, gm = G.gravity_force_vjp_batch(P, M, C, offs, workspace=ws, stats=sv, **kw)
        return f, gx, gm, G.stats_dict(sf), G.stats_dict(sv)

    f0, gx0, gm0, sf0, sv0 = run(ws)
    assert sf0["groups"] > 8 and sf0["far"] > 0 and sf0["near"] > 0
    assert torch.isfinite(gx0).all() and (f0 != 0).any(1).all()
    junk = torch.randint(0, 256, ws.shape, dtype=torch.uint8, device="cuda",
                         generator=torch.Generator(device="cuda").manual_seed(1))
    # on the costs of the walks before, on random bytes, and on costs and tags
    # that a walk of fewer groups left
    smaller = make().zero_()
    k = offs[-2] if len(sizes) > 1 else 690000
    G.gravity_force(P[:k].contiguous(), M[:k].contiguous(), workspace=smaller, **kw)
    for w in (ws, ws, junk, junk, smaller):
        f, gx, gm, sf, sv = run(w)
        assert torch.equal(f, f0) and sf == sf0 and sv == sv0
        # gradients: float atomics in arrival order
        for a, b in ((gx, gx0), (gm, gm0)):
            assert ((a - b).double().norm() / b.double().norm()).item() < 1e-5


# Adjoints of 3,000,000 points and more in all go by single waves too, every group
# of every set, and by cost: the walk leaves its costs' tag (a mark, then the
# number of groups) in the workspace for the next one.
@pytest.mark.parametrize("sizes,order", [((3000000,), 3), ((1690000, 690000, 65, 620011), 1),
                                         ((1690000, 690000, 65, 620011), 2)])
def test_large_adjoints_are_ordered_by_cost(gpu, sizes, order):
    G = _G()
    n = sum(sizes)
    P, M, C = (torch.cat(t) for t in zip(*(_points(k, k) for k in sizes)))
    offs = G.set_offsets(sizes)
    ws = G.new_batch_workspace(n, len(sizes), 10, 32).zero_()
    runs = []
    for _ in range(3):
        st = G.new_stats()
        gx, gm = G.gravity_force_vjp_batch(P, M, C, offs, softening_scale=0.005, leaf_size=32,
                                           multipole_order=order, workspace=ws, stats=st)
        runs.append((gx, gm, G.stats_dict(st)))
    words = ws[: ws.numel() // 4 * 4].view(torch.int32)
    tags = words[1:][words[:-1] == 0x5C4ED01E]
    assert runs[0][2]["groups"] in tags.tolist()
    for gx, gm, st in runs[1:]:
        assert st == runs[0][2]
        for a, b in ((gx, runs[0][0]), (gm, runs[0][1])):
            assert ((a - b).double().norm() / b.double().norm()).item() < 1e-5
