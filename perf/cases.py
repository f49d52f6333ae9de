"""Performance cases of the Barnes-Hut library: what its users run, through
the public entry points of sbh_amd, from a call of a few hundred points to the
largest configurations of the benchmark.

    listed()              the named cases
    draw(rng)             one more case of the same ranges
    prepare(case, seed)   inputs, and the workspace a program keeps, on the GPU
    run(state)            one pass; returns its whole outputs
    exact(case, seed)     the same outputs by direct sums in 64 bits
    work(case)            bytes and operations that one pass cannot do without
    tolerance(case)       how far another correct implementation may be off

Families ("path" of a case):
    gravity     adaptive-tree self-gravity: forces alone (a simulation step),
                or forces and the recompute adjoint through torch.autograd (a
                training step); orders 1/2 forward, 1/2/3 adjoint
    batch       many independent sets of uneven sizes in one forest
    direct      the exact sums: fwd + full adjoint of a small self-gravitating
                set, or forces of many sources at few queries, with or without
                the short-range cutoff and the periodic box
    octree8     the drop-in path over dense octree8 records: the recompute
                custom VJP, and the short-range TreePM force (periodic, cutoff,
                pruned) with its tree build
    wn          winding numbers of an oriented surface at many query points
    stochastic  the control-variate estimator on the adaptive tree
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "barnes-hut_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from sbh_amd import ffi, gravity, stochastic, wn  # noqa: E402

INF = float("inf")


# ------------------------------------------------------------------ cases
def _gravity(kind, n, leaf, eps, fwd, adj, **kw):
    return dict(path="gravity", kind=kind, n=n, leaf=leaf, eps=eps, fwd=fwd, adj=adj, **kw)


def listed():
    return [
        # forces of a small cluster, default options (quadrupole): latency and
        # launches decide
        _gravity("plummer", 2003, 32, 0.01, 2, 0, name="force_plummer_2003"),
        # the reference benchmark's size: 10,000 uniform points, fwd + adjoint
        _gravity("uniform", 10000, 16, 0.01, 1, 3, name="step_uniform_10000"),
        # default orders of the autograd wrapper (quadrupole both ways) at an
        # odd middle size
        _gravity("blobs", 100003, 32, 0.005, 2, 2, name="step_blobs_100003_quadrupole"),
        # custom-VJP configuration: 2^18 points in Gaussian blobs
        _gravity("blobs", 262144, 32, 0.002, 1, 3, name="step_blobs_262144"),
        # the headline: 2^20 Plummer points, fwd + adjoint
        _gravity("plummer", 1048576, 32, 0.005, 1, 3, name="step_plummer_1048576"),
        # uneven sets in one launch, fwd + adjoint (monopole, quadrupole, leaf
        # 24: what the autotuner picks for such batches)
        dict(path="batch", sets=48, lo=1024, hi=131072, leaf=24, eps=0.005, fwd=1, adj=2,
             name="batch_48_sets"),
        # exact self-gravity step at the reference benchmark's size
        dict(path="direct", mode="step", n=10000, m=10000, rc=INF, box=0.0, eps=0.01,
             name="direct_step_10000"),
        # exact short-range forces in a periodic box at some queries (the
        # check of a TreePM run)
        dict(path="direct", mode="force", n=65536, m=4099, rc=0.05, box=1.0, eps=0.002,
             name="direct_force_65536_at_4099"),
        # the drop-in custom VJP over octree8 records (builds and walks both
        # ways)
        dict(path="octree8", mode="step", n=100003, depth=7, rc=INF, eps=0.05, beta=2.0,
             name="octree8_step_100003"),
        # short-range TreePM force of a 128^3 particle mesh: build and walk
        dict(path="octree8", mode="treepm", n=128 ** 3, depth=8, rc=1.0, eps=0.1, beta=1.7,
             name="octree8_treepm_2097152"),
        # winding numbers of a closed surface at a million points
        dict(path="wn", n=204020, m=1048576, leaf=16, name="wn_204020_at_1048576"),
        # one control-variate sample per subdomain, every point a query
        dict(path="stochastic", n=262144, leaf=32, eps=0.005, name="stochastic_262144"),
    ]


def _size(rng, lo, hi):
    """A size spread over the logarithm of [lo, hi], odd more often than not."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return min(hi, max(lo, n | 1 if rng.random() < 0.7 else n))


def draw(rng):
    path = rng.choice(["gravity"] * 5 + ["batch", "direct", "direct", "octree8", "octree8", "wn",
                                        "stochastic"])
    if path == "gravity":
        fwd, adj = rng.choice([(1, 0), (2, 0), (1, 3), (1, 3), (2, 2), (1, 2), (1, 1), (2, 3)])
        hi = 1048576 if (fwd, adj) in ((1, 0), (2, 0), (1, 1), (1, 3)) else 400000
        return _gravity(rng.choice(["plummer", "uniform", "blobs"]), _size(rng, 500, hi),
                        rng.choice([16, 24, 32]), rng.choice([0.002, 0.005, 0.01]), fwd, adj)
    if path == "batch":
        fwd, adj = rng.choice([(1, 3), (1, 2), (2, 2)])
        return dict(path="batch", sets=rng.randint(3, 48), lo=rng.choice([200, 1024]),
                    hi=_size(rng, 8192, 131072), leaf=rng.choice([16, 24, 32]), eps=0.005,
                    fwd=fwd, adj=adj)
    if path == "direct":
        rc, box = rng.choice([(INF, 0.0), (INF, 0.0), (0.05, 0.0), (0.05, 1.0)])
        if rng.random() < 0.5:
            n = _size(rng, 300, 32768)
            return dict(path="direct", mode="step", n=n, m=n, rc=rc, box=box, eps=0.01)
        return dict(path="direct", mode="force", n=_size(rng, 1000, 262144),
                    m=_size(rng, 64, 16384), rc=rc, box=box, eps=0.002)
    if path == "octree8":
        if rng.random() < 0.5:
            return dict(path="octree8", mode="step", n=_size(rng, 1000, 262144),
                        depth=rng.choice([5, 6, 7]), rc=rng.choice([INF, 0.5]), eps=0.05,
                        beta=rng.choice([1.7, 2.0]))
        side = rng.randint(24, 128)
        return dict(path="octree8", mode="treepm", n=side ** 3, depth=6 if side <= 48 else 7
                    if side <= 80 else 8, rc=1.0, eps=0.1, beta=1.7)
    if path == "wn":
        return dict(path="wn", n=_size(rng, 1000, 204020), m=_size(rng, 1000, 1048576),
                    leaf=rng.choice([8, 16, 32]))
    return dict(path="stochastic", n=_size(rng, 4000, 524288), leaf=rng.choice([16, 32]),
                eps=0.005)


# ------------------------------------------------------------------ inputs
def _points(kind, n, g):
    """(points, masses): a Plummer sphere (a = 1, truncated at r = 20), a
    uniform unit cube, or 64 Gaussian blobs with log-normal masses."""
    if kind == "plummer":
        x_max = 20.0 ** 3 / (20.0 ** 2 + 1.0) ** 1.5
        x = torch.rand(n, generator=g, device="cuda", dtype=torch.float64) * x_max
        r = (x.clamp_min(1e-12) ** (-2.0 / 3.0) - 1.0) ** -0.5
        v = torch.randn((n, 3), generator=g, device="cuda", dtype=torch.float64)
        p = v * (r / v.norm(dim=1))[:, None]
        return p.float(), torch.full((n,), 1.0 / n, device="cuda")
    if kind == "uniform":
        p = torch.rand((n, 3), generator=g, device="cuda")
        return p, torch.full((n,), 1.0 / n, device="cuda")
    return _blobs(n, 64, g)


def _blobs(n, k, g):
    centres = torch.rand((k, 3), generator=g, device="cuda")
    which = torch.randint(k, (n,), generator=g, device="cuda")
    p = centres[which] + 0.02 * torch.randn((n, 3), generator=g, device="cuda")
    m = torch.exp(0.5 * torch.randn(n, generator=g, device="cuda"))
    return p, m / m.sum()


def _surface(n, g):
    """Oriented area elements of a closed star-shaped surface: n nearly even
    directions u (a Fibonacci lattice), radius 1 + sum a_k sin(w_k . u + f_k);
    centroids, outward unit normals and areas."""
    i = torch.arange(n, device="cuda", dtype=torch.float64) + 0.5
    z = 1.0 - 2.0 * i / n
    phi = math.pi * (1.0 + 5.0 ** 0.5) * i
    s = torch.sqrt(1.0 - z * z)
    u = torch.stack([s * torch.cos(phi), s * torch.sin(phi), z], 1)
    w = 2.0 * torch.randn((8, 3), generator=g, device="cuda", dtype=torch.float64)
    f = 2.0 * math.pi * torch.rand(8, generator=g, device="cuda", dtype=torch.float64)
    a = 0.03 * torch.randn(8, generator=g, device="cuda", dtype=torch.float64)
    t = u @ w.T + f
    r = 1.0 + torch.sin(t) @ a
    grad = (torch.cos(t) * a) @ w
    grad = grad - (grad * u).sum(1, keepdim=True) * u
    nrm = u - grad / r[:, None]
    nrm = nrm / nrm.norm(dim=1, keepdim=True)
    area = r * r / (nrm * u).sum(1) * (4.0 * math.pi / n)
    return (u * r[:, None]).float(), nrm.float(), area.float()


def _treepm(n, g):
    """side^3 particles in a periodic box of `side` cells: a displaced grid
    with 30% of the particles moved into Gaussian halos; masses 1."""
    side = round(n ** (1.0 / 3.0))
    axis = torch.arange(side, device="cuda", dtype=torch.float32)
    p = torch.stack(torch.meshgrid(axis, axis, axis, indexing="ij"), -1).reshape(-1, 3)
    p = p + 0.3 * torch.randn(p.shape, generator=g, device="cuda")
    k = int(0.3 * n)
    halos = max(8, n // 1000)
    which = torch.randint(halos, (k,), generator=g, device="cuda")
    centres = side * torch.rand((halos, 3), generator=g, device="cuda")
    p[torch.randperm(n, generator=g, device="cuda")[:k]] = \
        centres[which] + 0.5 * torch.randn((k, 3), generator=g, device="cuda")
    p = torch.remainder(p, float(side))
    p[p >= side] = 0.0
    return p.contiguous(), torch.ones(n, device="cuda"), float(side)


def _batch_sizes(case):
    """Set sizes, log-uniform in [lo, hi] (one from each of `sets` equal parts
    of the logarithm) in a mixed order; the same for every seed."""
    k = case["sets"]
    g = torch.Generator().manual_seed(1000 * k + case["hi"])
    t = (torch.arange(k, dtype=torch.float64) +
         torch.rand(k, generator=g, dtype=torch.float64)) / k
    lo, hi = math.log(case["lo"]), math.log(case["hi"])
    s = torch.exp(lo + (hi - lo) * t).round().long().tolist()
    order = torch.randperm(k, generator=g).tolist()
    return [s[i] for i in order]


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    path = case["path"]
    st = dict(case=case)
    if path == "gravity":
        n = case["n"]
        p, m = _points(case["kind"], n, g)
        st.update(p=p, m=m, ws=gravity.new_workspace(n, 10, case["leaf"]))
        if case["adj"]:
            p.requires_grad_(True)
            m.requires_grad_(True)
            st["c"] = torch.randn((n, 3), generator=g, device="cuda")
    elif path == "batch":
        sizes = _batch_sizes(case)
        sets = [_blobs(n, 8 + i % 57, g) for i, n in enumerate(sizes)]
        n = sum(sizes)
        st.update(p=torch.cat([s[0] for s in sets]), m=torch.cat([s[1] for s in sets]),
                  c=torch.randn((n, 3), generator=g, device="cuda"),
                  offs=gravity.set_offsets(sizes),
                  ws=gravity.new_batch_workspace(n, len(sizes), 10, case["leaf"]))
    elif path == "direct":
        p, m = _points("uniform", case["n"], g)
        st.update(p=p, m=m)
        if case["mode"] == "step":
            p.requires_grad_(True)
            m.requires_grad_(True)
            st["c"] = torch.randn((case["n"], 3), generator=g, device="cuda")
        else:
            st["q"] = torch.rand((case["m"], 3), generator=g, device="cuda")
    elif path == "octree8":
        if case["mode"] == "step":
            p, m = _points("plummer", case["n"], g)
            p.requires_grad_(True)
            m.requires_grad_(True)
            st.update(p=p, m=m, c=torch.randn((case["n"], 3), generator=g, device="cuda"))
        else:
            p, m, box = _treepm(case["n"], g)
            st.update(p=p, m=m, box=box, z=torch.zeros_like(p),
                      lo=torch.zeros(3, device="cuda"), hi=torch.full((3,), box, device="cuda"))
    elif path == "wn":
        p, nv, a = _surface(case["n"], g)
        q = 3.0 * torch.rand((case["m"], 3), generator=g, device="cuda") - 1.5
        st.update(p=p, nv=nv, a=a, q=q, ws=wn.new_workspace(case["n"], case["m"], 10,
                                                            case["leaf"]))
    else:
        p, m = _points("plummer", case["n"], g)
        st.update(p=p, m=m, seed=seed & 0x7fffffff,
                  ws=stochastic.new_workspace(case["n"], case["n"], 10, case["leaf"]))
    return st


# ------------------------------------------------------------------ one pass
def run(st):
    case = st["case"]
    path = case["path"]
    if path == "gravity":
        kw = dict(beta=2.0, softening_scale=case["eps"], max_depth=10, leaf_size=case["leaf"],
                  multipole_order=case["fwd"], workspace=st["ws"])
        if not case["adj"]:
            return gravity.gravity_force(st["p"], st["m"], **kw)
        f = gravity.gravity_force_recompute_vjp(st["p"], st["m"],
                                                vjp_multipole_order=case["adj"], **kw)
        gx, gm = torch.autograd.grad(f, (st["p"], st["m"]), grad_outputs=st["c"])
        return dict(f=f, gx=gx, gm=gm)
    if path == "batch":
        kw = dict(beta=2.0, softening_scale=case["eps"], max_depth=10, leaf_size=case["leaf"],
                  workspace=st["ws"], check_offsets=False)
        f = gravity.gravity_force_batch(st["p"], st["m"], st["offs"],
                                        multipole_order=case["fwd"], **kw)
        gx, gm = gravity.gravity_force_vjp_batch(st["p"], st["m"], st["c"], st["offs"],
                                                 multipole_order=case["adj"], **kw)
        return dict(f=f, gx=gx, gm=gm)
    if path == "direct":
        kw = dict(softening_scale=case["eps"], cutoff_scale=case["rc"],
                  periodic=case["box"] > 0.0, box_length=case["box"] or 1.0)
        if case["mode"] == "force":
            return ffi.softened_direct_force(st["p"], st["m"], st["q"], **kw)
        f = ffi.softened_direct_force_recompute_vjp(st["p"], st["m"], vjp_mode="full", **kw)
        gx, gm = torch.autograd.grad(f, (st["p"], st["m"]), grad_outputs=st["c"])
        return dict(f=f, gx=gx, gm=gm)
    if path == "octree8":
        if case["mode"] == "step":
            f = ffi.softened_barnes_hut_force_octree8_recompute_vjp(
                st["p"], st["m"], beta=case["beta"], softening_scale=case["eps"],
                cutoff_scale=case["rc"], max_depth=case["depth"])
            gx, gm = torch.autograd.grad(f, (st["p"], st["m"]), grad_outputs=st["c"])
            return dict(f=f, gx=gx, gm=gm)
        leaf, node = ffi.build_octree8_buffers(st["p"], st["z"], st["m"], st["lo"], st["hi"],
                                               max_depth=case["depth"])
        return ffi.softened_barnes_hut_force_octree8(
            leaf, node, st["p"], beta=case["beta"], softening_scale=case["eps"],
            cutoff_scale=case["rc"], prune_enabled=True, prune_r_cut_mult=4.0, periodic=True,
            box_length=st["box"])
    if path == "wn":
        return wn.winding_number(st["p"], st["nv"], st["a"], st["q"], beta=2.0, max_depth=10,
                                 leaf_size=case["leaf"], workspace=st["ws"])
    return stochastic.stochastic_gravity_force(
        st["p"], st["m"], st["p"], beta=2.0, samples_per_subdomain=1, seed=st["seed"],
        softening_scale=case["eps"], max_depth=10, leaf_size=case["leaf"], workspace=st["ws"])


# ------------------------------------------------------------------ 64 bits
_PAIRS = 1 << 24  # pairs per chunk of the direct sums


def _pair(q, p, eps, rc, box):
    """Of the pairs (query, source): displacement d, att s^3 and
    3 att s^5 + cutoff term (the softened, optionally attenuated kernel)."""
    d = q[:, None, :] - p[None]
    if box:
        d = d - box * torch.round(d / box)
    r2 = (d * d).sum(-1)
    s = (r2 + eps * eps + 1e-12) ** -0.5
    s3 = s ** 3
    if not math.isfinite(rc):
        return d, s3, 3.0 * s3 * s * s
    r = torch.sqrt(r2 + 1e-12)
    u = r / (2.0 * rc)
    e = torch.exp(-u * u)
    att = torch.special.erfc(u) + (2.0 / math.sqrt(math.pi)) * u * e
    cut = s3 * r * e / (2.0 * math.sqrt(math.pi) * rc ** 3)
    return d, att * s3, 3.0 * att * s3 * s * s + cut


def _direct(p, m, q, eps, rc=INF, box=0.0, c=None, full=False):
    """Forces at q; with c also the query-side gradient J^T c, or (full, q = p)
    the position and mass gradients of sum c . F.  All in 64 bits."""
    f, gx, gm = [], [], []
    step = max(1, _PAIRS // max(1, p.shape[0]))
    for a in range(0, q.shape[0], step):
        d, lin, k = _pair(q[a:a + step], p, eps, rc, box)
        f.append(-((m * lin)[..., None] * d).sum(1))
        if c is None:
            continue
        ck = c[a:a + step]
        u = (d * ck[:, None, :]).sum(-1)
        own = -(m * lin).sum(1)[:, None] * ck + ((m * k * u)[..., None] * d).sum(1)
        if full:
            v = (d * c[None]).sum(-1)
            other = -(lin @ c) + ((k * v)[..., None] * d).sum(1)
            gx.append(own - m[a:a + step, None] * other)
            gm.append((lin * v).sum(1))
        else:
            gx.append(own)
    out = dict(f=torch.cat(f))
    if c is not None:
        out["gx"] = torch.cat(gx)
        out["gm"] = torch.cat(gm) if full else torch.zeros_like(m)
    return out


def exact(case, seed):
    """The direct sums in 64 bits (the tree paths approximate them); None where
    they take too long, and for the random estimator."""
    path = case["path"]
    if path == "stochastic":
        return None
    if path == "batch":
        if sum(n * n for n in _batch_sizes(case)) > 1.5e10:
            return None
    elif case["n"] * case.get("m", case["n"]) > 1.5e10:
        return None
    st = prepare(case, seed)
    p, m = st["p"].detach().double(), (st["a"] if path == "wn" else st["m"]).detach().double()
    c = st["c"].double() if "c" in st else None
    if path == "gravity":
        r = _direct(p, m, p, case["eps"], c=c, full=True)
        return r if case["adj"] else r["f"]
    if path == "batch":
        rows = [0] + torch.cumsum(torch.tensor(_batch_sizes(case)), 0).tolist()
        parts = [_direct(p[a:b], m[a:b], p[a:b], case["eps"], c=c[a:b], full=True)
                 for a, b in zip(rows, rows[1:])]
        return {k: torch.cat([r[k] for r in parts]) for k in ("f", "gx", "gm")}
    if path == "direct":
        if case["mode"] == "step":
            return _direct(p, m, p, case["eps"], case["rc"], case["box"], c, True)
        return _direct(p, m, st["q"].double(), case["eps"], case["rc"], case["box"])["f"]
    if path == "octree8":
        if case["mode"] == "step":
            return _direct(p, m, p, case["eps"], case["rc"], 0.0, c)
        return _direct(p, m, p, case["eps"], case["rc"], st["box"])["f"]
    q, w = st["q"].double(), st["nv"].double() * m[:, None]
    out = []
    step = max(1, _PAIRS // case["n"])
    for a in range(0, q.shape[0], step):
        d = p[None] - q[a:a + step, None, :]
        r = d.norm(dim=-1)
        out.append(((d * w[None]).sum(-1) / (4.0 * math.pi * (r ** 3 + 1e-5))).sum(1))
    return torch.cat(out)


# ------------------------------------------------------------------ work
def _interactions(n, leaf, beta=2.0):
    """Interactions per query of a walk with MAC distance >= beta diagonals:
    per level the cells between beta diagonals of their own size and of their
    parents' (at most all of the level's), and the leaves nearer than that."""
    ball = 4.0 / 3.0 * math.pi * (beta * math.sqrt(3.0)) ** 3
    total, cells = 0.0, 8.0
    while n / cells > leaf / 2.0:
        total += min(cells, 7.0 * ball)
        cells *= 8.0
    return min(float(n), total + ball * leaf / 2.0)


def work(case):
    path = case["path"]
    if path == "batch":
        sizes = _batch_sizes(case)
        n = sum(sizes)
        pairs = sum(s * _interactions(s, case["leaf"]) for s in sizes)
        return dict(bytes=n * (16 + 12 + 28 + 16), flops=pairs * (20 + 48))
    n = case["n"]
    if path == "gravity":
        pairs = n * _interactions(n, case["leaf"])
        if case["adj"]:
            return dict(bytes=n * (28 + 28 + 16), flops=pairs * (20 + 48))
        return dict(bytes=n * 28, flops=pairs * 20)
    if path == "direct":
        pair = 20 if not math.isfinite(case["rc"]) else 45
        if case["mode"] == "step":
            return dict(bytes=n * (28 + 28 + 16), flops=float(n) * n * (2.4 * pair + pair))
        return dict(bytes=16 * n + 24 * case["m"], flops=float(n) * case["m"] * pair)
    if path == "octree8":
        nodes = (8 ** (case["depth"] + 1) - 1) // 7
        if case["mode"] == "step":
            pairs = n * _interactions(n, 8, case["beta"])
            return dict(bytes=2 * nodes * 136 + 2 * n * 48 + n * (28 + 40),
                        flops=pairs * (20 + 34))
        # particles within the prune radius of 4 cutoffs (one particle a cell)
        pairs = n * 4.0 / 3.0 * math.pi * (4.0 * case["rc"]) ** 3
        return dict(bytes=nodes * 136 + n * (28 + 32 + 12), flops=pairs * 45)
    if path == "wn":
        return dict(bytes=28 * n + 16 * case["m"],
                    flops=case["m"] * _interactions(n ** 0.75, case["leaf"]) * 20.0)
    return dict(bytes=n * 28, flops=n * _interactions(n, case["leaf"]) * 4.0)


def tolerance(case):
    """32-bit sums of thousands of terms over the same interactions: about four
    times the distance from the same sums in 64 bits (gravity forces 5e-7 to
    3e-6 and gradients up to 2.7e-6, single values of close pairs up to 6e-4;
    octree8 5e-6; direct sums 1.8e-6; winding numbers 2.5e-7)."""
    path = case["path"]
    if path in ("gravity", "batch"):
        return dict(rel=1.2e-5, max=2.2e-3)
    if path == "octree8":
        return dict(rel=2e-5, max=1e-3)
    if path == "direct":
        return dict(rel=8e-6, max=5e-4)
    if path == "wn":
        return dict(rel=2e-6, max=1e-4)
    # stochastic: differences of node and children sums, weighted by up to 1e4
    return dict(rel=8e-4, max=0.1)
