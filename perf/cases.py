"""The work that programs on this framework have it do, as timed cases.

Each case is one pass through a public entry point with what its caller has in hand already:
particles on the device (or, where the entry point takes host data, on the host), a solver
context, an embedding and its P matrix, a trained network. Sizes and settings are those of
bench.py, the tests and the reference's own drivers.

kinds of pass
  step        set_particles (device arrays), build, forces into device arrays: one force
              evaluation of a simulation whose state lives elsewhere in the program
  plugin      NBodySolverHipBH.updateTree + solveNbody on host points: the solver plug-in
              interface, as the t-SNE driver of the reference calls it
  leapfrog    set_particles, a few kick-drift-kick steps with a rebuild each, state read back
  batched     set_particles, build, forces of many independent systems in one context
  tsne        embedding set, a few iterations of the t-SNE descent, embedding read back
  cost        the KL divergence of an embedding (FP64, exact Z)
  learned     build, forces with the learned far-field correction, read back
  affinities  the t-SNE input affinities of host points, into the caller's arrays
  train       Adam steps of the far-field network on a labelled data set
"""
import ctypes
import math

import numpy as np
import torch

from masterthesislucas_amd import BHContext, _lib
from masterthesislucas_amd import tsne as T
from masterthesislucas_amd.learned import FarFieldMLP
from masterthesislucas_amd.solver import NBodySolverHipBH, Points

EPS = 1e-3   # Plummer softening of the gravity workloads
DT = 1e-4
# pairs up to which exact() sums every pair in FP64 (about ten seconds)
EXACT_PAIRS = 4.0e11


def listed():
    return [
        # a small N-body problem called in a loop: a handful of launches on an idle chip
        dict(name="step_2k", kind="step", n=2000, dist="disk", theta=0.5, tree="quadtree",
             total=False),
        # the headline workload: two Plummer disks, one force evaluation with its rebuild
        dict(name="step_1m", kind="step", n=1048576, dist="two_disks", theta=0.5,
             tree="quadtree", total=False),
        # the reference's solver plug-in on host points (fixed-depth Morton tree, bounds given),
        # at an odd count
        dict(name="plugin_20k", kind="plugin", n=20011, theta=0.5, tree="morton_fixed"),
        # a time integration between two snapshots
        dict(name="leapfrog_200k", kind="leapfrog", n=200003, dist="two_disks", theta=0.5,
             steps=8, graph=False),
        # many independent systems of very different size (even ones uniform disks, odd ones
        # Plummer disks), walked heaviest entries first
        dict(name="batched_128", kind="batched", systems=128, nmin=1024, nmax=65536, theta=0.5),
        # t-SNE at the size of MNIST: compact clusters early in the run, the spread embedding late
        dict(name="tsne_70k_early", kind="tsne", n=70000, phase="early", solver="bh", theta=0.5,
             iters=5),
        dict(name="tsne_70k_late", kind="tsne", n=70000, phase="late", solver="bh", theta=0.5,
             iters=5),
        # the same with the symmetric dual-tree FMM
        dict(name="tsne_fmm_70k", kind="tsne", n=70000, phase="late", solver="fmm_sym", theta=0.5,
             iters=5),
        # the cost a t-SNE program prints every so often
        dict(name="cost_70k", kind="cost", n=70000, phase="late"),
        # a large Plummer disk at an open angle with the learned correction
        dict(name="learned_4m", kind="learned", n=4194304, theta=0.9, terms=7),
        # t-SNE preprocessing: 784 pixels, perplexity 30, k = 90
        dict(name="affinities_20k", kind="affinities", n=20000, dim=784, perplexity=30.0, k=90),
        # training of the network: forward, backward, Adam
        dict(name="train_256k", kind="train", samples=262144, batch=4096, epochs=1, terms=7),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "plugin", "leapfrog", "batched", "tsne", "tsne",
                       "cost", "learned", "affinities", "train"])
    theta = round(rng.uniform(0.4, 1.0), 3)
    if kind == "step":
        # (the fixed-depth tree is for points without far outliers)
        tree, dist = rng.choice([("quadtree", "disk"), ("quadtree", "two_disks"),
                                 ("quadtree", "plummer"), ("morton_fixed", "disk")])
        return dict(kind=kind, n=_log_int(rng, 1000, 1048575), dist=dist, theta=theta, tree=tree,
                    total=rng.random() < 0.3)
    if kind == "plugin":
        return dict(kind=kind, n=_log_int(rng, 1000, 100000), theta=theta,
                    tree=rng.choice(["quadtree", "morton_fixed"]))
    if kind == "leapfrog":
        return dict(kind=kind, n=_log_int(rng, 1000, 500000), dist=rng.choice(["disk", "two_disks"]),
                    theta=theta, steps=rng.randint(2, 12), graph=rng.random() < 0.5)
    if kind == "batched":
        return dict(kind=kind, systems=rng.randint(8, 192), nmin=1024,
                    nmax=_log_int(rng, 4096, 65536), theta=theta)
    if kind == "tsne":
        return dict(kind=kind, n=_log_int(rng, 2000, 70000), phase=rng.choice(["early", "late"]),
                    solver=rng.choice(["bh", "bh", "fmm_sym"]), theta=theta,
                    iters=rng.randint(2, 8))
    if kind == "cost":
        return dict(kind=kind, n=_log_int(rng, 2000, 70000), phase=rng.choice(["early", "late"]))
    if kind == "learned":
        return dict(kind=kind, n=_log_int(rng, 50000, 2000000), theta=round(rng.uniform(0.7, 1.1), 3),
                    terms=rng.choice([3, 7]))
    if kind == "affinities":
        k = rng.randint(15, 120)
        return dict(kind=kind, n=_log_int(rng, 1000, 20000), dim=_log_int(rng, 20, 1000),
                    perplexity=round(k / 3.0, 2), k=k)
    return dict(kind=kind, samples=_log_int(rng, 8192, 262144),
                batch=rng.choice([1024, 4096, 16384]), epochs=1, terms=rng.choice([3, 7]))


# ---------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _rand(g, n):
    return torch.rand(n, generator=g, device="cuda", dtype=torch.float64)


def _plummer_radii(g, n, a):
    u = _rand(g, n)
    return a * torch.sqrt(u / (1.0 - u))


def _particles(dist, n, seed):
    """x, y, m, vx, vy on the device: a uniform disk at rest, a Plummer disk at rest, or two
    counter-rotating Plummer disks on circular orbits (total mass 1)."""
    g = _gen(seed)
    if dist == "disk":
        r, phi = torch.sqrt(_rand(g, n)), 2.0 * math.pi * _rand(g, n)
        x, y = r * torch.cos(phi), r * torch.sin(phi)
        vx, vy = torch.zeros_like(x), torch.zeros_like(x)
    elif dist == "plummer":
        r, phi = _plummer_radii(g, n, 1.0), 2.0 * math.pi * _rand(g, n)
        x, y = r * torch.cos(phi), r * torch.sin(phi)
        vx, vy = torch.zeros_like(x), torch.zeros_like(x)
    else:
        r, phi = _plummer_radii(g, n, 0.1), 2.0 * math.pi * _rand(g, n)
        s = torch.ones(n, device="cuda", dtype=torch.float64)
        s[: n // 2] = -1.0
        menc = 0.5 * r * r / (r * r + 0.01)
        vc = torch.sqrt(menc * r * r / (r * r + EPS * EPS) ** 1.5)
        x, y = 0.5 * s + r * torch.cos(phi), r * torch.sin(phi)
        vx, vy = s * vc * torch.sin(phi), -s * vc * torch.cos(phi)
    m = torch.full_like(x, 1.0 / n)
    return [t.to(torch.float32).contiguous() for t in (x, y, m, vx, vy)]


def _sizes(case):
    """Log-uniform sizes, the same for every seed (a program's context is made for its sizes)."""
    rng = np.random.default_rng([case["systems"], case["nmax"]])
    return np.floor(np.exp(rng.uniform(math.log(case["nmin"]), math.log(case["nmax"] + 1),
                                       case["systems"]))).astype(np.int64)


def _batch(case, seed):
    sizes = _sizes(case)
    n = int(sizes.sum())
    g = _gen(seed)
    odd = torch.repeat_interleave(torch.arange(sizes.size, device="cuda") % 2,
                                  torch.as_tensor(sizes, device="cuda"))
    phi = 2.0 * math.pi * _rand(g, n)
    r = torch.where(odd == 1, _plummer_radii(g, n, 0.1), torch.sqrt(_rand(g, n)))
    m = torch.repeat_interleave(1.0 / torch.as_tensor(sizes, device="cuda", dtype=torch.float64),
                                torch.as_tensor(sizes, device="cuda"))
    xyz = [t.to(torch.float32).contiguous() for t in (r * torch.cos(phi), r * torch.sin(phi), m)]
    return sizes, xyz


def _embedding(case, seed):
    """Ten clusters of 2-D points in shuffled order: compact ones around the origin with some
    points between them (early exaggeration), or discs that fill the plane (late)."""
    n = case["n"]
    rng = np.random.default_rng(seed)
    lab = rng.integers(0, 10, n)
    if case["phase"] == "early":
        c = rng.normal(0.0, 2.0, (10, 2))
        y = c[lab] + rng.normal(0.0, 0.05, (n, 2))
        stray = rng.random(n) < 0.1
        y[stray] = rng.normal(0.0, 2.0, (int(stray.sum()), 2))
    else:
        a = 2.0 * math.pi * np.arange(10) / 10.0
        c = 55.0 * np.stack([np.cos(a), np.sin(a)], 1) * (0.55 + 0.45 * (np.arange(10) % 2))[:, None]
        r, phi = 17.0 * np.sqrt(rng.random(n)), 2.0 * math.pi * rng.random(n)
        y = c[lab] + np.stack([r * np.cos(phi), r * np.sin(phi)], 1)
    return np.ascontiguousarray(y.astype(np.float32)), lab


def _affinity_graph(y, lab, seed):
    """A symmetric P over the points (CSR sorted by row and column, sum 1): 60 neighbours each
    way among the points next to a point in its cluster's order along a line through the plane,
    values spread as Gaussian affinities."""
    n = y.shape[0]
    rng = np.random.default_rng(seed + 1)
    order = torch.as_tensor(np.lexsort((y[:, 0] + 0.05 * y[:, 1], lab)), device="cuda")
    offs = np.sort(rng.choice(np.arange(1, 121), size=min(60, n // 3), replace=False))
    g = _gen(seed + 2)
    rows, cols, vals = [], [], []
    for o in offs:
        i, j = order[:-int(o)], order[int(o):]
        v = torch.exp(-4.0 * torch.rand(i.numel(), generator=g, device="cuda"))
        rows += [i, j]
        cols += [j, i]
        vals += [v, v]
    rows, cols, vals = torch.cat(rows), torch.cat(cols), torch.cat(vals)
    key, at = torch.sort(rows * n + cols)
    vals = (vals[at].double() / vals.double().sum()).to(torch.float32)
    ptr = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    ptr[1:] = torch.cumsum(torch.bincount(key // n, minlength=n), 0)
    return (ptr.cpu().numpy().astype(np.uint32), (key % n).cpu().numpy().astype(np.uint32),
            vals.cpu().numpy())


def _mixture(n, dim, seed):
    g = _gen(seed)
    means = 2.0 * torch.randn(10, dim, generator=g, device="cuda")
    lab = torch.randint(0, 10, (n,), generator=g, device="cuda")
    return (means[lab] + torch.randn(n, dim, generator=g, device="cuda")).cpu().numpy()


def _samples(n, seed):
    """Cell features with a unit direction and an opening ratio, and smooth labels of them."""
    rng = np.random.default_rng(seed)
    phi = 2.0 * math.pi * rng.random(n)
    X = np.concatenate([rng.normal(0.0, 0.1, (n, 10)), np.cos(phi)[:, None],
                        np.sin(phi)[:, None], rng.uniform(0.1, 0.9, (n, 1))], 1)
    w = np.exp(1j * phi)
    t = (0.7 + X[:, 0]) * w + (X[:, 1] + 1j * X[:, 2]) * w.conj() + 0.3 * X[:, 12] * w ** 3
    T_ = np.stack([t.real, t.imag], 1) + rng.normal(0.0, 0.01, (n, 2))
    return X.astype(np.float32), T_.astype(np.float32)


def _weights(seed):
    """A network as training starts it: uniform weights within 1/sqrt(fan in), zero biases."""
    rng = np.random.default_rng(seed + 3)
    out = []
    for i, o in ((10, 64), (64, 64), (64, 14)):
        out += [rng.uniform(-1.0, 1.0, i * o) / math.sqrt(i), np.zeros(o)]
    return np.concatenate(out).astype(np.float32)


def _ptr(a):
    return a.ctypes.data_as(ctypes.c_void_p)


# ---------------------------------------------------------------------------------------------
# passes
# ---------------------------------------------------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    st = dict(case=case)
    if kind in ("step", "leapfrog", "learned"):
        n = case["n"]
        st["p"] = _particles(case.get("dist", "plummer"), n, seed)
        st["ctx"] = BHContext(n, kernel="gravity", tree_mode=case.get("tree", "quadtree"),
                              softening=EPS)
        st["a"] = [torch.empty(n, device="cuda") for _ in range(2)]
        if kind == "learned":
            st["ctx"].learned_enable(True)
            st["net"] = FarFieldMLP(max_samples=1024, seed=seed)
            st["net"].terms = case["terms"]
            st["net"].set_params(0.1 * _weights(seed))
    elif kind == "plugin":
        y, _ = _embedding(dict(n=case["n"], phase="late"), seed)
        st["points"] = Points(y)
        st["solver"] = NBodySolverHipBH(kernel="tsne", theta=case["theta"], n_max=case["n"],
                                        tree_mode=case["tree"])
    elif kind == "batched":
        sizes, st["p"] = _batch(case, seed)
        n = int(sizes.sum())
        st["a"] = [torch.empty(n, device="cuda") for _ in range(2)]
        st["ctx"] = BHContext(n, kernel="gravity", softening=EPS, sizes=sizes)
        torch.cuda.synchronize()
        st["ctx"].set_particles(*st["p"])
        st["ctx"].build()
        st["ctx"].forces_device_only(case["theta"])
        st["ctx"].order_by_cost()
    elif kind in ("tsne", "cost"):
        y, lab = _embedding(case, seed)
        st["y"] = (np.ascontiguousarray(y[:, 0]), np.ascontiguousarray(y[:, 1]))
        theta = case.get("theta", 0.5)
        st["tsne"] = T.TSNE(*_affinity_graph(y, lab, seed), st["y"], min_theta=theta,
                            max_theta=theta, solver=case.get("solver", "bh"))
    elif kind == "affinities":
        n, k = case["n"], case["k"]
        st["X"] = _mixture(n, case["dim"], seed)
        st["ctx"] = BHContext(n, kernel="tsne")
        st["out"] = [np.zeros(n + 1, np.uint32), np.zeros(2 * n * k, np.uint32),
                     np.zeros(2 * n * k, np.float32), np.zeros((n, k), np.uint32),
                     np.zeros((n, k), np.float64), np.zeros(n, np.float64)]
    else:
        st["net"] = FarFieldMLP(max_samples=case["samples"], seed=seed)
        st["net"].terms = case["terms"]
        st["net"].set_dataset(*_samples(case["samples"], seed))
        st["w"] = _weights(seed)
    torch.cuda.synchronize()
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "step":
        ctx, (ax, ay) = st["ctx"], st["a"]
        ctx.set_particles(*st["p"][:3])
        ctx.build()
        total = ctx.forces_device(case["theta"], ax, ay, want_total=case["total"])
        return [ax, ay, total] if case["total"] else [ax, ay]
    if kind == "plugin":
        pts, sol = st["points"], st["solver"]
        pts.derivative[:] = 0.0
        sol.updateTree(pts, pts.position.min(0), pts.position.max(0))
        return [sol.solveNbody(pts), pts.derivative]
    if kind == "leapfrog":
        ctx = st["ctx"]
        ctx.set_particles(*st["p"])
        (ctx.leapfrog_graph if case["graph"] else ctx.leapfrog)(case["steps"], DT, case["theta"])
        return list(ctx.get_particles())
    if kind == "batched":
        ctx, (ax, ay) = st["ctx"], st["a"]
        ctx.set_particles(*st["p"])
        ctx.build()
        ctx.forces_device(case["theta"], ax, ay)
        return [ax, ay]
    if kind == "tsne":
        t = st["tsne"]
        t.ctx._c(_lib.load().bh_tsne_set_embedding(t.ctx.handle, _ptr(st["y"][0]),
                                                   _ptr(st["y"][1])))
        t.iteration_counter = 0 if case["phase"] == "early" else 500
        t.run(case["iters"])
        return t.embeddedPoints
    if kind == "cost":
        return list(st["tsne"].costFunction())
    if kind == "learned":
        ctx = st["ctx"]
        ctx.set_particles(*st["p"][:3])
        ctx.build()
        return list(ctx.forces_learned(st["net"], case["theta"])[:2])
    if kind == "affinities":
        ctx, (rp, col, val, idx, d2, beta), nnz = st["ctx"], st["out"], ctypes.c_uint32(0)
        ctx._c(_lib.load().bh_tsne_affinities(
            ctx.handle, _ptr(st["X"]), case["n"], case["dim"], case["perplexity"], case["k"],
            _ptr(rp), _ptr(col), _ptr(val), ctypes.byref(nnz), _ptr(idx), _ptr(d2), _ptr(beta)))
        return [rp, col, val, idx, d2, beta, nnz.value]
    net = st["net"]
    net.set_params(st["w"])
    loss = net.train(case["epochs"], batch=case["batch"], lr=2e-3, seed=7)
    return [loss, net.get_params()]


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------
def _walk_flops(n, theta, per=14.0):
    """A Barnes-Hut evaluation: about 2.5 / theta^1.6 cells and leaf particles accepted per
    particle and level of the tree, 14 or 15 operations each."""
    return per * n * 14.0 / theta ** 1.6 * max(1.0, math.log2(max(n, 32) / 16.0) / 2.0) * 1.2


def work(case):
    kind, n = case["kind"], case.get("n", 0)
    if kind == "step":
        return dict(bytes=20.0 * n, flops=_walk_flops(n, case["theta"]))
    if kind == "plugin":
        return dict(bytes=40.0 * n, flops=_walk_flops(n, case["theta"], 15.0))
    if kind == "leapfrog":
        return dict(bytes=36.0 * n * case["steps"], flops=(case["steps"] + 1) *
                    _walk_flops(n, case["theta"]))
    if kind == "batched":
        mean = (case["nmax"] - case["nmin"]) / math.log(case["nmax"] / case["nmin"])
        return dict(bytes=20.0 * mean * case["systems"],
                    flops=case["systems"] * _walk_flops(mean, case["theta"]))
    if kind == "tsne":
        nnz = 120.0 * n
        return dict(bytes=case["iters"] * (8.0 * nnz + 24.0 * n),
                    flops=case["iters"] * (_walk_flops(n, case["theta"], 15.0) + 10.0 * nnz))
    if kind == "cost":
        return dict(bytes=8.0 * 120.0 * n + 8.0 * n, flops=8.0 * n * n)
    if kind == "learned":
        return dict(bytes=20.0 * n, flops=_walk_flops(n, case["theta"]) * 2.5)
    if kind == "affinities":
        return dict(bytes=4.0 * n * case["dim"] + 24.0 * n * case["k"],
                    flops=2.0 * n * n * case["dim"])
    steps = case["samples"] // case["batch"] * case["epochs"]
    return dict(bytes=60.0 * case["samples"], flops=6.0 * 5632.0 * steps * case["batch"]
                + 2.0 * 5632.0 * case["samples"])


# ---------------------------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------------------------
def _sums(x, y, m, kernel):
    """Every pair in FP64: gravity accelerations and potentials, or the t-SNE repulsion and the
    per-point terms of Z (self excluded)."""
    n = x.numel()
    ax, ay, tot = (torch.empty(n, device="cuda", dtype=torch.float64) for _ in range(3))
    rows = max(1, int(2.0e8) // n)
    for a in range(0, n, rows):
        b = min(a + rows, n)
        dx, dy = x[None, :] - x[a:b, None], y[None, :] - y[a:b, None]
        d2 = dx * dx + dy * dy
        if kernel == "gravity":
            w = torch.rsqrt(d2 + float(np.float32(EPS)) ** 2)
            tot[a:b] = -(w @ m) + m[a:b] / float(np.float32(EPS))
            w = w * w * w * m[None, :]
            ax[a:b], ay[a:b] = (w * dx).sum(1), (w * dy).sum(1)
        else:
            w = 1.0 / (1.0 + d2)
            tot[a:b] = w.sum(1) - 1.0
            w = w * w
            ax[a:b], ay[a:b] = -(w * dx).sum(1), -(w * dy).sum(1)
    return ax, ay, tot


def _attraction(y, ptr, col, val):
    """Row sums of P_ij w_ij (y_j - y_i)."""
    n = y.shape[0]
    row = torch.repeat_interleave(torch.arange(n, device="cuda"), ptr[1:] - ptr[:-1])
    d = y[col] - y[row]
    w = val / (1.0 + (d * d).sum(1))
    return torch.zeros_like(y).index_add_(0, row, w[:, None] * d)


def _csr(y, lab, seed):
    ptr, col, val = _affinity_graph(y, lab, seed)
    return (torch.as_tensor(ptr.astype(np.int64), device="cuda"),
            torch.as_tensor(col.astype(np.int64), device="cuda"),
            torch.as_tensor(val.astype(np.float64), device="cuda"))


def _exact_train(case, seed):
    """Full-batch Adam in FP64 (with smaller batches the order is the library's own)."""
    if case["batch"] < case["samples"]:
        return None
    X, Tn = (torch.as_tensor(a.astype(np.float64), device="cuda")
             for a in _samples(case["samples"], seed))
    p = torch.as_tensor(_weights(seed).astype(np.float64), device="cuda").requires_grad_()

    def loss():
        o, h = 0, X[:, :10]
        for k, (i, j) in enumerate(((10, 64), (64, 64), (64, 14))):
            h = h @ p[o:o + i * j].reshape(i, j) + p[o + i * j:o + i * j + j]
            o += i * j + j
            h = torch.nn.functional.silu(h) if k < 2 else h
        w = torch.complex(X[:, 10], X[:, 11])
        q = X[:, 12]
        b = [w, w.conj(), w ** 3, q + 0j, q * w ** 2, q * w.conj() ** 2, q * w ** 4]
        s = sum(torch.complex(h[:, 2 * t], h[:, 2 * t + 1]) * b[t] for t in range(case["terms"]))
        return ((s.real - Tn[:, 0]) ** 2 + (s.imag - Tn[:, 1]) ** 2).sum() / (2.0 * len(q))

    opt = torch.optim.Adam([p], lr=2e-3, betas=(0.9, 0.999), eps=1e-8)
    for _ in range(case["epochs"]):
        opt.zero_grad()
        loss().backward()
        opt.step()
    return [loss().item(), p.detach()]


def _exact_affinities(case, seed):
    n, k = case["n"], case["k"]
    X = torch.as_tensor(_mixture(n, case["dim"], seed).astype(np.float64), device="cuda")
    sq = (X * X).sum(1)
    d2, idx = torch.empty(n, k, device="cuda", dtype=torch.float64), None
    idx = torch.empty(n, k, device="cuda", dtype=torch.int64)
    for a in range(0, n, 2048):
        b = min(a + 2048, n)
        d = sq[a:b, None] + sq[None, :] - 2.0 * (X[a:b] @ X.t())
        d[torch.arange(b - a, device="cuda"), torch.arange(a, b, device="cuda")] = math.inf
        idx[a:b] = torch.topk(d, k, dim=1, largest=False).indices
        e = X[idx[a:b].reshape(-1)].reshape(b - a, k, -1) - X[a:b, None, :]
        e = (e * e).sum(2)
        e, at = torch.sort(e, dim=1)
        d2[a:b], idx[a:b] = e, torch.gather(idx[a:b], 1, at)
    dr = d2 - d2[:, :1]
    beta = torch.ones(n, device="cuda", dtype=torch.float64)
    lo, hi = torch.full_like(beta, -math.inf), torch.full_like(beta, math.inf)
    live = torch.ones(n, device="cuda", dtype=torch.bool)
    P = torch.zeros_like(dr)
    for _ in range(200):
        e = torch.exp(-beta[:, None] * dr)
        s = e.sum(1)
        p = e / s[:, None]
        diff = torch.log(s) + beta * (dr * p).sum(1) - math.log(case["perplexity"])
        P[live] = p[live]
        live = live & (diff.abs() >= 1e-5)
        if not bool(live.any()):
            break
        up = live & (diff > 0)
        down = live & ~(diff > 0)
        lo, hi = torch.where(up, beta, lo), torch.where(down, beta, hi)
        beta = torch.where(up, torch.where(torch.isinf(hi), beta * 2.0, 0.5 * (beta + hi)),
                           torch.where(down, torch.where(torch.isinf(lo), beta * 0.5,
                                                         0.5 * (beta + lo)), beta))
    row = torch.arange(n, device="cuda")[:, None].expand(n, k)
    key = torch.cat([(row * n + idx).reshape(-1), (idx * n + row).reshape(-1)])
    uniq, inv = torch.unique(key, return_inverse=True)
    val = torch.zeros(uniq.numel(), device="cuda", dtype=torch.float64)
    val.index_add_(0, inv, torch.cat([P.reshape(-1), P.reshape(-1)]) / (2.0 * n))
    val = torch.nn.functional.pad(val, (0, 2 * n * k - val.numel()))
    return [None, None, val, None, d2, beta, None]


def exact(case, seed):
    kind = case["kind"]
    if kind in ("step", "leapfrog", "learned"):
        n, steps = case["n"], case.get("steps", 0)
        if float(n) * n * (steps + 1) > EXACT_PAIRS:
            return None
        x, y, m, vx, vy = (t.double() for t in _particles(case.get("dist", "plummer"), n, seed))
        ax, ay, phi = _sums(x, y, m, "gravity")
        if kind == "leapfrog":
            dt = float(np.float32(DT))
            for _ in range(steps):
                vx, vy = vx + 0.5 * dt * ax, vy + 0.5 * dt * ay
                x, y = x + dt * vx, y + dt * vy
                ax, ay, _ = _sums(x, y, m, "gravity")
                vx, vy = vx + 0.5 * dt * ax, vy + 0.5 * dt * ay
            return [x, y, vx, vy]
        return [ax, ay, float(phi.sum())] if case.get("total") else [ax, ay]
    if kind == "plugin":
        y, _ = _embedding(dict(n=case["n"], phase="late"), seed)
        y = torch.as_tensor(y.astype(np.float64), device="cuda")
        ax, ay, tot = _sums(y[:, 0].contiguous(), y[:, 1].contiguous(), None, "tsne")
        return [float(tot.sum()), torch.stack([ax, ay], 1)]
    if kind == "batched":
        sizes, (x, y, m) = _batch(case, seed)
        if float((sizes.astype(np.float64) ** 2).sum()) > EXACT_PAIRS:
            return None
        got, o = [], 0
        for s in sizes:
            got.append(_sums(*(t[o:o + int(s)].double() for t in (x, y, m)), "gravity")[:2])
            o += int(s)
        return [torch.cat([a[k] for a in got]) for k in (0, 1)]
    if kind in ("tsne", "cost"):
        y, lab = _embedding(case, seed)
        ptr, col, val = _csr(y, lab, seed)
        y = torch.as_tensor(y.astype(np.float64), device="cuda")
        if kind == "cost":
            z = _sums(y[:, 0].contiguous(), y[:, 1].contiguous(), None, "tsne")[2].sum()
            row = torch.repeat_interleave(torch.arange(case["n"], device="cuda"),
                                          ptr[1:] - ptr[:-1])
            d = y[col] - y[row]
            q = 1.0 / (1.0 + (d * d).sum(1)) / z
            return [float((val * torch.log2(val / q)).sum()), float(z)]
        early = case["phase"] == "early"
        exag, mu = (16.0, 0.5) if early else (4.0, 0.8)
        prev = y
        for _ in range(case["iters"]):
            rx, ry, tot = _sums(y[:, 0].contiguous(), y[:, 1].contiguous(), None, "tsne")
            d = 4.0 / tot.sum() * torch.stack([rx, ry], 1) + exag * _attraction(y, ptr, col, val)
            y, prev = y + case["n"] / 15.0 * d + mu * (y - prev), y
        return y
    if kind == "affinities":
        return _exact_affinities(case, seed)
    return _exact_train(case, seed)
