"""Kernels at the edges of their tiles: remainders, the smallest sizes, and sizes past one tile
or one launch's blocks, each against the FP64 oracle or plain numpy."""
import numpy as np
import pytest

from masterthesislucas_amd import BHContext, tsne
from masterthesislucas_amd.learned import N_OUT, FarFieldMLP, flatten, unflatten
from oracle import oracle as O
from tests.helpers import oracle_tree, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("terms", [3, 7])
@pytest.mark.parametrize("n", [1, 31, 32, 33, 100, 256 * 32 + 5])
def test_training_gradient_edges(gpu, n, terms):
    """Samples in tiles of 32, at most 256 tiles at a time: one sample, around one tile, a ragged
    last tile, and a block that takes two tiles. Gradient blocks to 1e-4 of their norm, as FP32
    activations with FP32 sums (n products of about 1e-7 relative error each) allow."""
    rng = np.random.default_rng(100 + n)
    p = {"W1": rng.normal(0, 0.4, (10, 64)), "b1": rng.normal(0, 0.1, 64),
         "W2": rng.normal(0, 0.15, (64, 64)), "b2": rng.normal(0, 0.1, 64),
         "W3": rng.normal(0, 0.15, (64, N_OUT)), "b3": rng.normal(0, 0.1, N_OUT)}
    p = {k: v.astype(np.float32) for k, v in p.items()}
    X = rng.normal(0, 1, (n, 13)).astype(np.float32)
    a = rng.uniform(0, 2 * np.pi, n)
    X[:, 10], X[:, 11] = np.cos(a), np.sin(a)
    X[:, 12] = rng.uniform(0.05, 1.0, n)
    T = rng.normal(0, 0.5, (n, 2)).astype(np.float32)
    net = FarFieldMLP(max_samples=max(n, 16))
    net.terms = terms
    net.set_params(flatten(p))
    loss, g = net.loss_grad(X, T)
    ref_loss, ref_g = O.learned_loss_grad(X.astype(np.float64), T.astype(np.float64),
                                          {k: v.astype(np.float64) for k, v in p.items()},
                                          terms=terms)
    assert abs(loss - ref_loss) < 1e-5 * ref_loss
    gg = unflatten(g)
    for k in ref_g:
        num = np.linalg.norm(gg[k].astype(np.float64) - ref_g[k])
        assert num < 1e-4 * np.linalg.norm(ref_g[k]) + 1e-9, k
    # the data-set loss that training reports (forward only) is the same loss
    net.set_dataset(X, T)
    assert abs(net.train(0) - ref_loss) < 1e-5 * ref_loss
    net.close()


@pytest.mark.parametrize("n", [2, 3, 255, 256, 257, 513, 1500])
def test_exact_z_edges(gpu, n):
    """Z over tiles of 256 x 256 pairs: less than a tile, exact tiles, ragged last tiles, with
    coincident and far points; Z and KL to 1e-12 (each of the n^2 FP64 terms carries a few units
    of 1e-16)."""
    rng = np.random.default_rng(n)
    y = rng.normal(0, 3, (n, 2)).astype(np.float32)
    y[-1] = y[0]
    if n > 2:
        y[1] = (3e4, -2e4)
    rows = np.repeat(np.arange(n), min(n - 1, 4))
    cols = (rows + 1 + np.tile(np.arange(min(n - 1, 4)), n)) % n
    o = np.lexsort((cols, rows))
    rows, cols = rows[o], cols[o]
    val = rng.uniform(0.1, 1.0, rows.size)
    val = (val / val.sum()).astype(np.float32)
    rp = np.zeros(n + 1, np.uint32)
    rp[1:] = np.cumsum(np.bincount(rows, minlength=n))
    t = tsne.TSNE(rp, cols.astype(np.uint32), val, (y[:, 0].copy(), y[:, 1].copy()))
    kl, z = t.costFunction()
    t.close()
    d = y.astype(np.float64)
    d2 = ((d[:, None, :] - d[None, :, :]) ** 2).sum(2)
    w = 1.0 / (1.0 + d2)
    np.fill_diagonal(w, 0.0)
    want_z = w.sum()
    p = val.astype(np.float64)
    want_kl = (p * np.log2(p * want_z * (1.0 + d2[rows, cols]))).sum()
    assert abs(z - want_z) <= 1e-12 * want_z
    assert abs(kl - want_kl) <= 1e-12 * np.abs(p * np.log2(p * want_z)).sum()


@pytest.mark.parametrize("n,dim,k", [(2, 1, 1), (129, 63, 5), (257, 64, 90), (513, 65, 128),
                                     (1100, 20, 30), (2600, 130, 15)])
def test_affinity_tile_edges(gpu, n, dim, k):
    """Row blocks of 128, column tiles of 256 in one or several ranges, K chunks of 64: the exact
    neighbours and distances against FP64 brute force (distances to 1e-12, as FP64 sums in another
    order allow; ties by index)."""
    rng = np.random.default_rng(n + dim)
    X = (rng.normal(0, 1, (n, dim)) + 3.0 * rng.integers(0, 4, (n, 1))).astype(np.float32)
    X[-1] = X[0]  # a duplicate pair
    a = tsne.affinities(X, perplexity=max(1.0, k / 3.0), k=k)
    d = X.astype(np.float64)
    d2 = ((d[:, None, :] - d[None, :, :]) ** 2).sum(2) if n * n * dim < 4e7 else None
    if d2 is None:
        d2 = np.stack([((d - row) ** 2).sum(1) for row in d])
    np.fill_diagonal(d2, np.inf)
    idx = np.argsort(d2, axis=1, kind="stable")[:, :k]
    want = np.take_along_axis(d2, idx, 1)
    assert np.allclose(a["d2"], want, rtol=1e-12, atol=0)
    differ = a["idx"] != idx  # only where two distances agree to rounding
    gap = np.abs(np.take_along_axis(d2, a["idx"].astype(np.int64), 1) - want)
    assert np.all(gap[differ] <= 1e-12 * want[differ])
    assert abs(a["val"].astype(np.float64).sum() - 1.0) < 1e-6


def _walk(p, kernel, theta, split, mode="quadtree", eps=1e-3, cap=16, want_total=True):
    from masterthesislucas_amd import BHContext
    ctx = BHContext(len(p[0]), kernel=kernel, tree_mode=mode, softening=eps, max_children=cap)
    ctx.set_particles(*p)
    ctx.set_split(split)
    ctx.build()
    ax, ay, tot = ctx.forces(theta, want_total=want_total)
    cnt = ctx.counters()
    return ctx, ax, ay, tot, cnt


def _points(case, n, rng):
    """x, y, masses: a disk; a tight cluster under a chain of one-child cells (a far outlier sets
    the root square); a line; points of which a third sit on one spot (a leaf of n / 3 at the
    depth limit)."""
    if case == "line":
        x, y = rng.uniform(-1, 1, n), np.zeros(n)
    else:
        r, a = np.sqrt(rng.random(n)), rng.uniform(0, 2 * np.pi, n)
        x, y = r * np.cos(a), r * np.sin(a)
    if case == "chain":
        x, y = 1e-5 * x, 1e-5 * y
        x[-1] = 900.0
    if case == "spot":
        x[: n // 3], y[: n // 3] = 0.25, 0.125
    m = rng.uniform(0.5, 1.5, n) / n
    return tuple(v.astype(np.float32) for v in (x, y, m))


@pytest.mark.parametrize("case", ["disk", "chain", "line", "spot"])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 129, 1000, 5000])
def test_walk_edges(gpu, case, n):
    """The walk at the edges of its sink groups (64), its source blocks (64, quads of 4) and its
    collected cells, on 1, 2 and 4 waves per group: bit-identical results and counts, and forces
    within the exact-walk bar of the FP64 sum of the same interactions (counts equal). A leaf of
    many coincident points sums them in plain FP32 batches: the bar holds there too."""
    from tests.helpers import check_exact_walk
    rng = np.random.default_rng(n)
    p = _points(case, n, rng)
    for theta in (0.5, 1.0):
        ctx, ax, ay, tot, cnt = _walk(p, "gravity", theta, 2)
        check_exact_walk(ctx, *p, "gravity", theta, float(np.float32(1e-3)), ax, ay, tot)
        ctx.close()
        for split in (1, 8):
            ctx, bx, by, tot2, cnt2 = _walk(p, "gravity", theta, split)
            ctx.close()
            assert np.array_equal(ax.view(np.uint32), bx.view(np.uint32))
            assert np.array_equal(ay.view(np.uint32), by.view(np.uint32))
            assert tot2 == tot and cnt2 == cnt


@pytest.mark.parametrize("n", [100, 1000, 70000])
def test_walk_small_opening_angle(gpu, n):
    """theta = 0.05 on few and many sinks: nearly every cell is opened, so the stack of opened
    cells fills and the walk falls back to one cell at a time; counts and forces as above."""
    from tests.helpers import check_exact_walk
    from masterthesislucas_amd.workloads import sample_indices
    rng = np.random.default_rng(7)
    p = _points("disk", n, rng)
    ctx, ax, ay, tot, cnt = _walk(p, "gravity", 0.05, 1, want_total=n <= 1000)
    if n <= 1000:
        check_exact_walk(ctx, *p, "gravity", 0.05, float(np.float32(1e-3)), ax, ay, tot)
    else:
        s = sample_indices(n, 256).astype(np.uint32)
        dx, dy, _ = ctx.direct_fp64(s)
        # the monopole error at l / r = 0.05 is about (l / r)^2 / 8 of a cell's pull
        assert np.quantile(np.hypot(ax[s] - dx, ay[s] - dy) / np.hypot(dx, dy), 0.9) < 1e-3
    ctx.close()


def test_walk_tsne_paths_agree(gpu):
    """The t-SNE sums of bh_forces (pre-order walk up to 131,072 points) and of the list walk
    (any split above 1) select the same interactions and differ by rounding only."""
    from tests.helpers import rel_err
    rng = np.random.default_rng(11)
    x, y, _ = _points("spot", 20011, rng)
    p = (20.0 * x, 20.0 * y, None)
    c1, ax, ay, z, cnt = _walk(p, "tsne", 0.5, 1)
    c2, bx, by, z2, cnt2 = _walk(p, "tsne", 0.5, 4)
    assert cnt == cnt2
    r = rel_err(bx, by, ax.astype(np.float64), ay.astype(np.float64))
    assert np.median(r) <= 1e-6 and np.quantile(r, 0.999) <= 1e-4
    assert abs(z2 - z) <= 1e-5 * z
    c1.close()
    c2.close()


def _check_sort(x, y, mode):
    n = len(x)
    xd, yd = x.astype(np.float64), y.astype(np.float64)
    minx, miny, maxx, maxy = xd.min(), yd.min(), xd.max(), yd.max()
    if mode == "quadtree":
        ref = O.morton64(xd, yd, minx, miny, O.quadtree_side(minx, miny, maxx, maxy), 32)
    else:
        ref = O.morton32(xd, yd, minx, miny, max(maxx + (-minx), maxy + (-miny))).astype(np.uint64)
    p = np.argsort(ref, kind="stable")
    ctx = BHContext(n, kernel="gravity", tree_mode=mode, softening=0.01)
    ctx.set_particles(x, y)
    ctx.build()
    codes, perm = ctx.morton()
    assert np.array_equal(perm, p)
    assert np.array_equal(codes, ref[p])
    ctx.close()


@pytest.mark.parametrize("mode", ["quadtree", "morton_fixed"])
@pytest.mark.parametrize("n", [2, 63, 64, 65, 1025, 8192, 8193, 10_241, 262_144, 524_288, 524_289,
                               1_048_577, 2_097_152, 2_097_153])
def test_sort_edges(gpu, mode, n):
    """Both sides of every size at which the sort changes its kernels or bucket size, one point
    in eight on one of three spots: codes and order bit-exact against a stable sort."""
    rng = np.random.default_rng(n)
    x, y = rng.normal(0, 1, (2, n)).astype(np.float32)
    dup = rng.random(n) < 1 / 8
    x[dup] = y[dup] = np.float32(0.25) * rng.integers(0, 3, dup.sum())
    _check_sort(x, y, mode)


@pytest.mark.parametrize("mode", ["quadtree", "morton_fixed"])
@pytest.mark.parametrize("low", ["spread", "equal"])
@pytest.mark.parametrize("n,mean", [(20_000, 512), (600_000, 1024)])
def test_sort_sample_misses_the_distribution(gpu, mode, low, n, mean):
    """Every key that the sort samples lies above every other key, so all the others fall into
    the first bucket, many times what one block sorts in LDS: still bit-exact."""
    b = -(-n // mean)
    s = b * next(q for q in (64, 32, 16, 8) if q == 8 or b * q <= 4096)
    j = np.arange(s, dtype=np.uint64)
    p0, p1 = n * j // s, n * (j + 1) // s
    h = (j * 0x9E3779B1) & 0xFFFFFFFF
    h ^= h >> 15
    h = (h * 0x85EBCA77) & 0xFFFFFFFF
    pick = p0 + ((h * (p1 - p0)) >> 32)
    rng = np.random.default_rng(n)
    t = rng.uniform(0, 0.5, n).astype(np.float32) if low == "spread" else np.zeros(n, np.float32)
    t[pick] = rng.uniform(0.75, 1.0, s).astype(np.float32)
    _check_sort(t, t.copy(), mode)


@pytest.mark.parametrize("mode", ["quadtree", "morton_fixed"])
@pytest.mark.parametrize("n", [1, 40, 700, 3000, 262_144, 262_145])
def test_node_moments_edges(gpu, mode, n):
    """Mass and centre of every node against FP64 prefix sums over the sorted particles, for trees
    of one chunk, of several, and on both sides of the size at which the chunks grow. A node's sum
    is at most 8 terms of a leaf batch after another and then 4 children per level: a relative
    error of about 100 x 2^-24 at most, 1e-5 with the centre's offsets measured in cell sides."""
    rng = np.random.default_rng(n + 1)
    x, y = rng.normal(0, 1, (2, n)).astype(np.float32)
    if n > 100:
        x[: n // 50] = y[: n // 50] = 0.5  # a crowded spot: a deep chain of cells, a large leaf
    m = rng.uniform(0.5, 1.5, n).astype(np.float32)
    ctx = BHContext(n, kernel="gravity", tree_mode=mode, softening=0.01)
    ctx.set_particles(x, y, m)
    ctx.build()
    _, perm = ctx.morton()
    t = ctx.tree()
    ctx.close()
    ms = m[perm].astype(np.float64)
    s0, sx, sy = (np.concatenate([[0.0], np.cumsum(v)])
                  for v in (ms, ms * x[perm].astype(np.float64), ms * y[perm].astype(np.float64)))
    f, e = t["first"].astype(np.int64), t["first"].astype(np.int64) + t["count"].astype(np.int64)
    assert f[0] == 0 and e[0] == n and t["skip"][0] == len(f)
    mass = s0[e] - s0[f]
    assert np.max(np.abs(t["mass"] - mass) / mass) < 1e-5
    extent = max(np.ptp(x), np.ptp(y), 1e-3)
    assert np.max(np.abs(t["cx"] - (sx[e] - sx[f]) / mass)) < 1e-5 * extent
    assert np.max(np.abs(t["cy"] - (sy[e] - sy[f]) / mass)) < 1e-5 * extent


@pytest.mark.parametrize("mode", ["quadtree", "morton_fixed"])
@pytest.mark.parametrize("n", [1, 17, 1023, 1024, 1025, 2049, 33_000])
def test_tree_emission_edges(gpu, mode, n):
    """Node numbering over tiles of 1024 particles, cells found near a particle, through the block's
    table of codes and by the wide search: every record equals the oracle's. A crowded spot gives
    long chains of single cells and leaves past the table's stride."""
    rng = np.random.default_rng(n + 2)
    x, y = rng.normal(0, 1, (2, n)).astype(np.float32)
    if n > 1000:
        x[: n // 3] = (0.5 + 1e-3 * rng.normal(0, 1, n // 3)).astype(np.float32)
        y[: n // 3] = (0.5 + 1e-3 * rng.normal(0, 1, n // 3)).astype(np.float32)
        x[: n // 20] = y[: n // 20] = np.float32(0.5)
    ctx = BHContext(n, kernel="gravity", tree_mode=mode, softening=0.01)
    ctx.set_particles(x, y)
    ctx.build()
    g = ctx.tree()
    ctx.close()
    t = oracle_tree(x, y, mode=mode)
    for k in ("level", "first", "count", "skip"):
        assert np.array_equal(g[k].astype(np.int64), t["tree"][k].astype(np.int64)), k
    assert np.array_equal((g["flags"] >> 1) & 1, t["pp"])


@pytest.mark.parametrize("n", [20_000, 100_000, 140_000])
def test_giant_cell_sums_in_order(gpu, n):
    """A cell with one child is a particle-particle cell; one that holds a whole cluster is summed
    in particle order in plain FP32 (1, 2 and 4 parts per wave). One source outweighs the others
    by 2^26, so a plain sum loses most of them and any other order would differ by about 1e-4;
    against the same sum in numpy to 2e-6 (terms to a few 2^-24)."""
    rng = np.random.default_rng(n)
    x, y = (0.30 + 0.02 * rng.random((2, n))).astype(np.float32)
    m = np.full(n, 2.0 ** -26, np.float32)
    x[0], y[0], m[0] = 0.30, 0.30, 1.0  # first in Morton order
    x[1], y[1] = 1.0, 1.0
    x[2], y[2] = 0.0, 0.0
    y[2], x[2] = 0.99, 0.0  # keeps the box at [0, 1]
    y[3], x[3] = 0.0, 0.99
    eps = float(np.float32(1e-3))
    ctx = BHContext(n, kernel="gravity", softening=eps)
    ctx.set_particles(x, y, m)
    ctx.build()
    fx, fy = ctx.forces(0.5)[:2]
    _, perm = ctx.morton()
    t = ctx.tree()
    ctx.close()
    giant = np.nonzero(((t["flags"] >> 1) & 1).astype(bool) & (t["count"] > 4096))[0][0]
    lo, hi = int(t["first"][giant]), int(t["first"][giant] + t["count"][giant])
    assert hi - lo > n - 8
    src = perm[lo:hi]
    sinks = src[rng.integers(1, hi - lo, 64)]
    f64, f32 = np.float64, np.float32
    px, py = x[sinks], y[sinks]
    gx, gy = np.zeros(64, f32), np.zeros(64, f32)
    eps2 = f32(eps) * f32(eps)
    for j in src:
        dx, dy = x[j] - px, y[j] - py
        d2 = (dx.astype(f64) ** 2 + (dy * dy).astype(f64)).astype(f32) + eps2
        inv = (1.0 / np.sqrt(d2.astype(f64))).astype(f32)
        g = m[j] * inv * inv * inv
        on = sinks != j
        gx = np.where(on, (gx.astype(f64) + g.astype(f64) * dx).astype(f32), gx)
        gy = np.where(on, (gy.astype(f64) + g.astype(f64) * dy).astype(f32), gy)
    # the few points outside the cell are far and light: below 1e-6 of the sums
    scale = np.hypot(gx, gy)
    assert np.max(np.abs(fx[sinks] - gx) / scale) < 2e-6
    assert np.max(np.abs(fy[sinks] - gy) / scale) < 2e-6


@pytest.mark.parametrize("n", [1, 5, 256, 257, 262_144, 262_145])
def test_velocities_through_builds(gpu, n):
    """The state that builds reorder, on both sides of the sizes at which the key kernel takes four
    particles per thread: positions and velocities come back in the caller's order and unchanged,
    velocities given, not given (zero), zero after given ones, and kicked from rest (dt a / 2
    before and after a drift that moves close pairs a little: within 5% of the largest dt a)."""
    rng = np.random.default_rng(n)
    x, y, vx, vy = rng.normal(0, 1, (4, n)).astype(np.float32)
    m = np.full(n, 1.0 / n, np.float32)
    ctx = BHContext(n, kernel="gravity", softening=0.05)
    for given in (True, False, True, False):
        ctx.set_particles(x, y, m, *((vx, vy) if given else ()))
        for _ in range(2):
            ctx.build()
        gx, gy, gu, gv = ctx.get_particles()
        assert np.array_equal(gx, x) and np.array_equal(gy, y)
        assert np.array_equal(gu, vx if given else 0 * vx)
        assert np.array_equal(gv, vy if given else 0 * vy)
    ax, ay, _ = ctx.forces(0.5)
    ctx.set_particles(x, y, m)
    ctx.leapfrog(1, 0.0, 0.5)  # no drift, no kick
    assert not np.any(ctx.get_particles()[2])
    dt = 2.0 ** -12
    ctx.set_particles(x, y, m)
    ctx.leapfrog(1, dt, 0.5)
    gx, gy, gu, gv = ctx.get_particles()
    ctx.build()
    hx, hy, hu, hv = ctx.get_particles()
    assert np.array_equal(gu, hu) and np.array_equal(gv, hv) and np.array_equal(gx, hx)
    top = max(np.abs(ax).max(), np.abs(ay).max(), 1e-30) * dt
    if n > 1:
        assert np.abs(gu - dt * ax).max() < 0.05 * top and np.any(gu)
    ctx.close()


@pytest.mark.parametrize("solver", ["bh", "fmm_sym"])
@pytest.mark.parametrize("n", [40, 256, 257, 5000, 262_400])
def test_tsne_run_equals_single_steps(gpu, solver, n):
    """Iterations in one call start from what the update before left (particles, bounds), single
    steps stage the embedding anew: the same embedding to the bit, through the change of the
    exaggeration, past one block and past the blocks that sum Z and take the bounds."""
    rng = np.random.default_rng(n)
    y = rng.normal(0, 1e-2, (n, 2)).astype(np.float32)
    cols = ((np.arange(n)[:, None] + np.array([1, 7, n - 7, n - 1])) % n).astype(np.uint32)
    cols.sort(axis=1)
    rp = (4 * np.arange(n + 1)).astype(np.uint32)
    val = np.full(4 * n, 1.0 / (4 * n), np.float32)
    out = []
    for single in (False, True):
        t = tsne.TSNE(rp, cols.ravel(), val, (y[:, 0].copy(), y[:, 1].copy()), solver=solver)
        t.iteration_counter = 247
        if single:
            zs = [t.timeStep() for _ in range(6)]
            assert all(np.isfinite(z) and z > 0 for z in zs)
        else:
            t.run(2)
            t.run(4)
        out.append(t.embeddedPoints)
        t.close()
    assert np.all(np.isfinite(out[0])) and np.any(out[0] != y)
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("theta", [0.35, 0.8])
@pytest.mark.parametrize("n", [64, 300, 4096, 16_384, 16_400, 66_000])
def test_fmm_edges(gpu, n, theta):
    """Leaf units at the edges of their lane groups (leaves of about 8, 16, 32 and many points side
    by side), units of more points than are staged at once, and trees whose leaf level is and is
    not among the levels of one block. FP64 on both sides, the order of the sums apart: FP32
    rounding of the result (median 1e-6, p99 1e-5), Z to 1e-10."""
    rng = np.random.default_rng(n)
    # four quadrants of densities 1 : 2 : 4 : 9, and a crowded spot
    q = np.searchsorted(np.cumsum([1, 2, 4, 9]) / 16, rng.random(n))
    x = (rng.random(n) + (q & 1)).astype(np.float32)
    y = (rng.random(n) + (q >> 1)).astype(np.float32)
    c = n // 40
    x[:c] = (0.3 + 1e-3 * rng.random(c)).astype(np.float32)
    y[:c] = (0.3 + 1e-3 * rng.random(c)).astype(np.float32)
    ctx = BHContext(n, kernel="tsne", tree_mode="morton_fixed")
    ctx.set_solver("fmm_sym")
    ctx.set_particles(x, y)
    ctx.build()
    ax, ay, z = ctx.forces(theta)
    ctx.close()
    t = oracle_tree(x, y, None, mode="morton_fixed")
    minx, miny, maxx, maxy = t["bounds"]
    tree = O.fixed_tree(t["xs"], t["ys"], t["depth"], minx, miny, maxx, maxy)
    sx, sy, bz = O.fmm_sym(t["xs"], t["ys"], tree, t["depth"], theta)
    bx, by = np.empty(n), np.empty(n)
    bx[t["perm"]], by[t["perm"]] = sx, sy
    r = rel_err(ax, ay, bx, by)
    assert np.median(r) <= 1e-6 and np.quantile(r, 0.99) <= 1e-5, (np.median(r), r.max())
    assert abs(z - bz) <= 1e-10 * abs(bz)


@pytest.mark.parametrize("n", [1, 1000, 4096, 4097, 262_200])
def test_leapfrog_steps_in_one_call(gpu, n):
    """Steps in one call share a launch between the closing kick of one and the opening kick and
    drift of the next, and hand the new positions' bounds to the build: the same state to the bit
    as one step per call and as replayed graphs, on both sides of the sizes at which the key kernel
    takes the bounds itself and at which the drift's blocks stop growing."""
    rng = np.random.default_rng(n)
    x, y, vx, vy = rng.normal(0, 1, (4, n)).astype(np.float32)
    m = np.full(n, 1.0 / n, np.float32)
    out = []
    for how in ("one", "single", "graph"):
        ctx = BHContext(n, kernel="gravity", softening=0.05)
        ctx.set_particles(x, y, m, vx, vy)
        if how == "one":
            ctx.leapfrog(3, 1e-2, 0.6)
        elif how == "single":
            for _ in range(3):
                ctx.leapfrog(1, 1e-2, 0.6)
        else:
            ctx.leapfrog_graph(3, 1e-2, 0.6)
        out.append(ctx.get_particles())
        ctx.close()
    for other in out[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(out[0], other))
    assert np.any(out[0][0] != x)


@pytest.mark.parametrize("order", ["far_first", "near_first"])
@pytest.mark.parametrize("n,dim,k", [(700, 64, 20), (3000, 33, 90)])
def test_affinity_thresholds_edges(gpu, n, dim, k, order):
    """Columns in order of distance, so that the first thresholds keep all or almost none of the
    later ones, and one point of ten times the others' norm, which loosens the short test of
    its columns: the exact neighbours against FP64 brute force, distances to 1e-12."""
    rng = np.random.default_rng(n)
    r = np.sort(rng.uniform(0.01, 1.0, n))[:, None]
    if order == "far_first":
        r = r[::-1]
    X = (r * rng.normal(0, 1, (n, dim))).astype(np.float32)
    X[n // 2] *= 10.0
    a = tsne.affinities(X, perplexity=k / 3.0, k=k)
    d = X.astype(np.float64)
    d2 = np.stack([((d - row) ** 2).sum(1) for row in d])
    np.fill_diagonal(d2, np.inf)
    want = np.sort(d2, axis=1)[:, :k]
    assert np.allclose(a["d2"], want, rtol=1e-12, atol=0)
    got = np.take_along_axis(d2, a["idx"].astype(np.int64), 1)
    assert np.allclose(got, want, rtol=1e-12, atol=0)


@pytest.mark.parametrize("kernel,n", [("gravity", 1), ("gravity", 64), ("gravity", 65),
                                      ("gravity", 20_001), ("gravity", 150_001), ("tsne", 300),
                                      ("tsne", 140_001)])
def test_forces_in_callers_order(gpu, kernel, n):
    """The walk (1, 2 and 4 parts per wave) and the pre-order walk store the forces in the caller's
    order: host and device outputs, both or one of them, are the same to the bit."""
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(n)
    x, y = rng.normal(0, 1, (2, n)).astype(np.float32)
    ctx = BHContext(n, kernel=kernel, softening=0.01)
    ctx.set_particles(x, y)
    ctx.build()
    ax, ay, _ = ctx.forces(0.5)
    _, perm = ctx.morton()
    for gx, gy in ((True, True), (True, False), (False, True)):
        dx, dy = (torch.full((n,), 7.0, device="cuda") for _ in range(2))
        torch.cuda.synchronize()
        ctx.forces_device(0.5, dx if gx else None, dy if gy else None)
        torch.cuda.synchronize()
        assert np.array_equal(dx.cpu().numpy(), ax if gx else np.full(n, 7.0, np.float32))
        assert np.array_equal(dy.cpu().numpy(), ay if gy else np.full(n, 7.0, np.float32))
    # another input order, the same tree: the same forces at the same points
    ctx.set_particles(x[perm], y[perm])
    ctx.build()
    bx, by, _ = ctx.forces(0.5)
    ctx.close()
    assert np.array_equal(bx, ax[perm]) and np.array_equal(by, ay[perm])


@pytest.mark.parametrize("sizes", [[1] * 256, [255, 1, 256, 257, 1, 1, 510, 2, 3],
                                   [300] + [2] * 120 + [1, 5, 1000, 31], [1024, 256, 256, 1]])
def test_batched_system_boundaries(gpu, sizes):
    """Many systems in one block of 256 particles, systems that start and end at a block's edge:
    every particle is in its own system. theta = 0 sums every pair: FP32 sums of at most 1000
    terms, a few times 6e-8 each, against FP64 direct sums."""
    rng = np.random.default_rng(len(sizes))
    n = sum(sizes)
    x, y = rng.normal(0, 1, (2, n)).astype(np.float32)
    m = rng.uniform(0.5, 1.5, n).astype(np.float32)
    ctx = BHContext(n, kernel="gravity", softening=0.01, sizes=sizes)
    ctx.set_particles(x, y, m)
    ctx.build()
    ax, ay, _ = ctx.forces(0.0)
    ctx.close()
    wx, wy, scale = np.zeros(n), np.zeros(n), np.zeros(n)
    o = 0
    for k in sizes:
        s = slice(o, o + k)
        dx = x[s].astype(np.float64)[None, :] - x[s].astype(np.float64)[:, None]
        dy = y[s].astype(np.float64)[None, :] - y[s].astype(np.float64)[:, None]
        w = m[s].astype(np.float64) / (dx * dx + dy * dy + float(np.float32(0.01)) ** 2) ** 1.5
        wx[s], wy[s] = (w * dx).sum(1), (w * dy).sum(1)
        scale[s] = (w * np.hypot(dx, dy)).sum(1)
        o += k
    assert np.all(np.abs(ax - wx) <= 2e-5 * scale)
    assert np.all(np.abs(ay - wy) <= 2e-5 * scale)


@pytest.mark.parametrize("n", [5 * 1024 * 64, 5 * 1024 * 64 + 1, 400_003])
@pytest.mark.parametrize("kernel,batched", [("gravity", False), ("gravity", True), ("tsne", False),
                                            ("tsne", True)])
def test_walk_resident_builds(gpu, kernel, batched, n):
    """Up to and past five sink groups per SIMD, where launches change to the walk held to fewer
    registers: the parts of a sink's sum are fixed, so forces, totals and counts equal those of two and
    four waves per group (always the other build) to the bit."""
    rng = np.random.default_rng(n)
    x, y = rng.normal(0, 1, (2, n)).astype(np.float32)
    kw = dict(sizes=[n // 3, 1, n - n // 3 - 1]) if batched else {}
    ctx = BHContext(n, kernel=kernel, softening=0.01, **kw)
    ctx.set_particles(x, y)
    ctx.build()
    for total in (False, True):
        got = []
        for split in (1, 2, 4):
            ctx.set_split(split)
            ax, ay, tot = ctx.forces(0.8, want_total=total)
            got.append((ax, ay, (tot, ctx.counters())))
        for ax, ay, rest in got[1:]:
            assert rest == got[0][2]
            assert np.array_equal(ax, got[0][0]) and np.array_equal(ay, got[0][1])
    ctx.close()


def test_training_gradient_of_many_samples(gpu):
    """The gradient of a batch of 4 million: a block's sums stay at 1,024 samples however many there
    are. All samples equal, so that a sum's roundings add up: a plain sum of m equal terms is off by at
    most m / 2 x 2^-24, so 1,024 samples, 4,096 / 16 partials and 16 sums of those by 3.9e-5; 1e-6 for
    the FP32 terms themselves."""
    n = 1 << 22
    rng = np.random.default_rng(5)
    p = {"W1": rng.normal(0, 0.4, (10, 64)), "b1": rng.normal(0, 0.1, 64),
         "W2": rng.normal(0, 0.15, (64, 64)), "b2": rng.normal(0, 0.1, 64),
         "W3": rng.normal(0, 0.15, (64, N_OUT)), "b3": rng.normal(0, 0.1, N_OUT)}
    p = {k: v.astype(np.float32) for k, v in p.items()}
    X = rng.normal(0, 1, (1, 13)).astype(np.float32)
    X[:, 10:] = (0.6, 0.8, 0.5)
    T = rng.normal(0, 0.5, (1, 2)).astype(np.float32)
    net = FarFieldMLP(max_samples=16)
    net.set_params(flatten(p))
    loss, g = net.loss_grad(np.tile(X, (n, 1)), np.tile(T, (n, 1)))
    net.close()
    ref_loss, ref = O.learned_loss_grad(X.astype(np.float64), T.astype(np.float64),
                                        {k: v.astype(np.float64) for k, v in p.items()}, terms=7)
    assert abs(loss - ref_loss) < 1e-5 * ref_loss
    g = unflatten(g)
    for k in ref:
        assert np.abs(g[k] - ref[k]).max() <= 4e-5 * np.abs(ref[k]).max(), k


@pytest.mark.parametrize("n,dim,k,kept", [(3000, 100, 30, True), (52_000, 1024, 128, False)])
def test_affinity_workspace_is_given_back(gpu, n, dim, k, kept):
    """The workspace of a call stays with the context up to 1 GiB and goes back with bh_tsne_set_p;
    a larger one (1.25 GB here) goes back with the call. Device memory as the driver counts it, to 64
    MiB (a context's own buffers do not change)."""
    torch = pytest.importorskip("torch")
    import ctypes as C

    from masterthesislucas_amd import _lib
    rng = np.random.default_rng(n)
    X = rng.standard_normal((n, dim), dtype=np.float32)
    ctx = BHContext(n, kernel="tsne")
    rp, col, val = (np.empty(m, t) for m, t in ((n + 1, np.uint32), (2 * n * k, np.uint32),
                                                (2 * n * k, np.float32)))
    ptr = lambda a: a.ctypes.data_as(C.c_void_p)  # noqa: E731
    nnz = C.c_uint32(0)
    before = torch.cuda.mem_get_info()[0]
    ctx._c(_lib.load().bh_tsne_affinities(ctx.handle, ptr(X), n, dim, k / 3.0, k, ptr(rp), ptr(col),
                                          ptr(val), C.byref(nnz), None, None, None))
    held = before - torch.cuda.mem_get_info()[0]
    print(f"held {held} bytes", flush=True)
    small = np.array([0, 1, 2], np.uint32)
    ctx._c(_lib.load().bh_tsne_set_p(ctx.handle, 2, ptr(small), ptr(np.array([1, 0], np.uint32)),
                                     ptr(np.full(2, 0.5, np.float32)), 2))
    after = before - torch.cuda.mem_get_info()[0]
    ctx.close()
    assert held < (1 << 30) + (64 << 20) if kept else held < 64 << 20
    assert after < 64 << 20
    assert rp[n] == nnz.value and np.all(np.diff(rp.astype(np.int64)) >= k)


@pytest.mark.parametrize("mode", ["quadtree", "morton_fixed"])
@pytest.mark.parametrize("n", [8192 * 1024, 8192 * 1024 + 1])
def test_tree_emission_of_many_tiles(gpu, mode, n):
    """Both sides of the 8,192 tiles up to which a block adds up the node counts of the tiles before
    its own; past them the counts are scanned first: every record equals the oracle's."""
    rng = np.random.default_rng(n)
    x, y = rng.normal(0, 1, (2, n)).astype(np.float32)
    ctx = BHContext(n, kernel="gravity", tree_mode=mode, softening=0.01)
    ctx.set_particles(x, y)
    ctx.build()
    g = ctx.tree()
    ctx.close()
    t = oracle_tree(x, y, mode=mode)
    for k in ("level", "first", "count", "skip"):
        assert np.array_equal(g[k].astype(np.int64), t["tree"][k].astype(np.int64)), k


def test_tree_emission_time_is_linear(gpu):
    """The tree's launches for 134 million particles take 8 times those for 17 million (9.3 measured;
    12.4 when every block added up the counts of all tiles before its own)."""
    torch = pytest.importorskip("torch")
    us = []
    for n in (1 << 24, 1 << 27):
        g = torch.Generator(device="cuda")
        g.manual_seed(1)
        x, y = (torch.randn(n, generator=g, device="cuda") for _ in range(2))
        torch.cuda.synchronize()
        ctx = BHContext(n, kernel="gravity", softening=1e-3)
        ctx.set_particles(x, y)
        del x, y
        ctx.build()
        ctx.profile_phases(["tree"])
        t = []
        for _ in range(5):
            ctx.profile_read(reset=True)
            ctx.build()
            t.append(ctx.profile_read(reset=True)["tree"][0])
        us.append(1e3 * np.median(t))
        ctx.close()
    torch.cuda.empty_cache()
    print(f"[tree] {us[0]:.0f} us, {us[1]:.0f} us", flush=True)
    assert us[1] < 11.0 * us[0], us
