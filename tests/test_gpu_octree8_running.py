"""octree8 walks over large clouds in shallow trees: each query's contributions
go to one running sum in the order of the reference's DFS (the last child first,
the points of a leaf in input order), rounding for rounding."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS, RC = 0.05, 2.0


def _terms(kind, q, g, p, m):
    """Contributions of the points to one query in 64 bits, (n, 3)."""
    d = q.astype(np.float64) - p.astype(np.float64)
    r2 = (d * d).sum(1)
    if kind == "grav":
        return -(m / (np.sqrt(r2) + 0.1) ** 3)[:, None] * d
    from scipy.special import erfc

    s = (r2 + EPS * EPS + 1e-12) ** -0.5
    lin, cc = s ** 3, 0.0
    if kind.endswith("cut"):
        r = np.sqrt(r2 + 1e-12)
        u = r / (2.0 * RC)
        e = np.exp(-u * u)
        cc = s ** 3 * r * e / (2.0 * np.sqrt(np.pi) * RC ** 3)
        lin = lin * (erfc(u) + 2.0 / np.sqrt(np.pi) * u * e)
    if kind.startswith("force"):
        return -(m * lin)[:, None] * d
    k = (d @ g.astype(np.float64)) * (3.0 * lin * s * s + cc)
    return -m[:, None] * (lin[:, None] * g - k[:, None] * d)


# first number of points with running sums: 98,304 at depth 5 with cutoff, twice
# that without, divided by 1.5 for each level less
@pytest.mark.parametrize("kind,depth,line", [("force_cut", 3, 43691), ("vjp_cut", 3, 43691),
                                             ("force", 2, 58255), ("grav", 1, 38837)])
@pytest.mark.parametrize("below", [False, True])
def test_sums_in_the_order_of_the_dfs(gpu, kind, depth, line, below):
    from sbh_amd import ffi

    n = line - 1 if below else line
    rng = np.random.default_rng(depth)
    # one heavy point in the octant that comes first, light ones (each below
    # half an ulp of its contribution) in the others, queries off the near corner
    p = rng.uniform(0.0, 1.0, (n, 3)).astype(np.float32)
    far = (p >= 0.5).all(1)
    p[far, rng.integers(0, 3, far.sum())] -= np.float32(0.5)
    p[7] = 0.9
    m = np.full(n, 1e-9, np.float32)
    m[7] = 1.0
    q = rng.uniform(-0.6, -0.4, (70, 3)).astype(np.float32)
    g = rng.uniform(0.5, 1.0, (70, 3)).astype(np.float32)
    leaf, node = ffi.build_octree8_buffers(p, np.zeros_like(p), m, min_corner=np.zeros(3, np.float32),
                                           max_corner=np.ones(3, np.float32), max_depth=depth)
    # beta = inf: every point is a term of every query
    soft = dict(beta=float("inf"), softening_scale=EPS, prune_enabled=False,
                cutoff_scale=RC if kind.endswith("cut") else float("inf"))
    if kind == "grav":
        out = ffi.barnes_hut_force_octree8(leaf, node, q, beta=float("inf"))
    elif kind.startswith("force"):
        out = ffi.softened_barnes_hut_force_octree8(leaf, node, q, **soft)
    else:
        out = ffi.softened_barnes_hut_force_octree8_vjp(leaf, node, q, g, **soft)
    out = out.cpu().numpy()
    cell = np.minimum((p * np.float32(1 << depth)).astype(np.int64), (1 << depth) - 1)
    code = sum(((cell[:, a] >> b) & 1) << (3 * b + a) for a in range(3) for b in range(depth))
    order = np.argsort(-code, kind="stable")
    whole, running = [], []
    for k in range(70):
        t = _terms(kind, q[k], g[k], p[order], m[order].astype(np.float64))
        whole.append(t.sum(0))
        running.append(np.add.accumulate(t.astype(np.float32), 0, dtype=np.float32)[-1])
    whole, running = np.array(whole), np.array(running, np.float64)
    rel = lambda a, b: np.linalg.norm(a - b) / np.linalg.norm(b)
    lost = rel(running, whole)
    assert lost > 2e-5  # of the light points, which the running sum loses
    if below:
        # partial sums keep most of them
        assert rel(out, whole) < 0.5 * lost
    else:
        # the one contribution that counts: about 10 roundings of 6e-8
        assert rel(out, running) < 6e-7
