"""Calls whose path depends on their size or input, on each path that the other tests leave out: the
radix sort's give-up, the affinity call that is repeated with one column range, the learned walk
with one, two and four waves per group and with totals, and captured steps after a change of what
they were captured with, and affinity calls that are refused or have the smallest inputs."""
import numpy as np
import pytest

from masterthesislucas_amd import BHContext, _lib, tsne
from masterthesislucas_amd._lib import BHError
from masterthesislucas_amd.learned import N_OUT, FarFieldMLP, flatten
from masterthesislucas_amd.workloads import two_plummer_disks
from oracle import oracle as O
from tests.helpers import WALK_TOL, exact_walk, oracle_tree
from tests.test_gpu_learned import _gpu_tree, _params, _plummer_ctx

pytestmark = pytest.mark.gpu

EPS = float(np.float32(1e-3))


@pytest.mark.parametrize("n", [20_000, 1 << 21, (1 << 21) + 1])
def test_sort_give_up_of_each_sort(gpu, n):
    """The bucket sort (up to 2^21 keys) and the radix sort (above) with a wait bound of 0 polls,
    set from the host: a build that gave up is reported and leaves no tree, one that did not is
    right, and with the default bound the order is bit-exact again."""
    p = two_plummer_disks(n, seed=33)
    ctx = BHContext(n, kernel="gravity", softening=EPS)
    ctx.set_particles(p.x, p.y, p.m)
    ctx.set_sort_spin_limit(0)
    raised = 0
    for _ in range(3):
        try:
            ctx.build()
        except BHError as e:
            assert e.status == _lib.BH_ERR_HIP and "look-back" in str(e)
            raised += 1
            with pytest.raises(BHError) as f:
                ctx.forces(0.5)
            assert f.value.status == _lib.BH_ERR_STATE
    # hundreds of tiles start together and some finds its predecessor unpublished; 10 tiles may not
    assert raised >= 1 or n == 20_000
    ctx.set_sort_spin_limit(1 << 22)
    ctx.build()
    codes, perm = ctx.morton()
    ctx.close()
    t = oracle_tree(p.x, p.y, p.m, mode="quadtree")
    assert np.array_equal(perm, t["perm"])
    assert np.array_equal(codes, t["codes_sorted"])


def test_affinities_repeated_with_one_range(gpu):
    """1,024 points are two column ranges of 512. The first 512 lie on a line along the first axis, the
    others on a ring around that axis, so that a point of the line has all of them at one distance:
    more than its list of the second range can hold beside each other, while one list over all
    columns has the near points of the line first and drops the ring. Neighbours exact, distances to
    1e-12."""
    rng = np.random.default_rng(5)
    n, dim, k = 1024, 64, 60
    X = np.zeros((n, dim))
    X[:512, 0] = np.linspace(-0.3, 0.3, 512)
    z = rng.normal(0, 1, (512, dim - 1))
    X[512:, 1:] = 0.5 * z / np.linalg.norm(z, axis=1, keepdims=True)
    X[512:, 0] = np.sqrt(0.75)
    X = X.astype(np.float32)
    a = tsne.affinities(X, perplexity=20.0, k=k)
    d = X.astype(np.float64)
    d2 = np.stack([((d - row) ** 2).sum(1) for row in d])
    np.fill_diagonal(d2, np.inf)
    want = np.sort(d2, axis=1)[:, :k]
    assert np.allclose(a["d2"], want, rtol=1e-12, atol=0)
    got = np.take_along_axis(d2, a["idx"].astype(np.int64), 1)
    assert np.allclose(got, want, rtol=1e-12, atol=0)
    # far points of the line from the ring: their distance agrees to 2^-11 of it and less
    ring = np.sqrt(d2[:512, 512:])
    assert np.all(np.ptp(ring, axis=1) < 2.0 ** -11 * ring.mean(axis=1))


@pytest.mark.parametrize("total", [False, True])
@pytest.mark.parametrize("n", [60_003, 100_003, 150_003, 400_003])
def test_learned_walk_of_each_launch(gpu, n, total):
    """Four, two and one wave per group and the build held to fewer registers, with and without the
    potential: constant coefficients (a last layer of zeros) against the FP64 walk on the GPU's
    tree; the potential is the plain walk's."""
    theta, band, terms = 0.9, 0.4, 7
    ctx, p = _plummer_ctx(n, seed=34)
    t = _gpu_tree(ctx, p)
    net = FarFieldMLP(max_samples=16)
    net.terms = terms
    prm = _params(35)
    prm["W3"][:] = 0.0
    prm["b3"][:] = np.random.default_rng(36).uniform(-1, 1, N_OUT).astype(np.float32)
    net.set_params(flatten(prm))
    ax, ay, pot = ctx.forces_learned(net, theta, band=band, want_total=total)
    pn, pp = ctx.counters()
    coef = np.broadcast_to(prm["b3"].astype(np.float64), (t["tree"]["first"].size, N_OUT))
    bx, by, cnt = O.bh_traverse_learned(t["xs"], t["ys"], t["ms"], t["tree"], t["side"],
                                        O.inv_theta2_f32(theta), coef, inv_band2=1.0 / band ** 2,
                                        eps2=EPS * EPS)
    w = exact_walk(ctx, p.x, p.y, p.m, "gravity", theta, eps=EPS)
    assert (int(pn), int(pp)) == (int(cnt[0]), int(cnt[1])) == (w["pn"], w["pp"])
    assert 0 < int(cnt[2]) < int(cnt[0])
    rx, ry = np.empty(n), np.empty(n)
    rx[t["perm"]], ry[t["perm"]] = bx, by
    # the bar of the exact walk scaled by the coefficients' size (test_learned_walk_matches_oracle)
    bar = WALK_TOL * (1.0 + 4.0 * np.abs(prm["b3"]).sum())
    assert np.max(np.abs(ax - rx) / w["abs_x"]) <= bar
    assert np.max(np.abs(ay - ry) / w["abs_y"]) <= bar
    if total:
        assert pot == ctx.forces(theta, want_total=True)[2]
    net.close()
    ctx.close()


@pytest.mark.parametrize("n1,n2", [(3000, 9001), (20_011, 700), (5000, 5000)])
def test_captured_steps_follow_the_particles(gpu, n1, n2):
    """Steps captured for one particle set and replayed after another was set, larger, smaller or of
    the same size: the state of eager steps to the bit, several replays long."""
    rng = np.random.default_rng(n1 + n2)
    ctx = BHContext(max(n1, n2), kernel="gravity", softening=0.05)
    for n in (n1, n2, n1):
        x, y, vx, vy = rng.normal(0, 1, (4, n)).astype(np.float32)
        m = np.full(n, 1.0 / n, np.float32)
        ctx.set_particles(x, y, m, vx, vy)
        ctx.leapfrog_graph(2, 1e-2, 0.6)
        ctx.leapfrog_graph(3, 1e-2, 0.6)
        got = ctx.get_particles()
        eager = BHContext(n, kernel="gravity", softening=0.05)
        eager.set_particles(x, y, m, vx, vy)
        eager.leapfrog(5, 1e-2, 0.6)
        want = eager.get_particles()
        eager.close()
        assert all(np.array_equal(a, b) for a, b in zip(got, want))
    ctx.close()


def test_captured_steps_follow_the_learned_switch(gpu):
    """Steps captured before the learned correction was switched on build no second moments; replayed
    after it they are captured anew: the cell features are those of eager steps."""
    n = 4000
    rng = np.random.default_rng(1)
    x, y, vx, vy = rng.normal(0, 1, (4, n)).astype(np.float32)
    m = np.full(n, 1.0 / n, np.float32)
    out = []
    for graph in (False, True):
        ctx = BHContext(n, kernel="gravity", softening=0.05)
        for on in (False, True):
            ctx.learned_enable(on)
            ctx.set_particles(x, y, m, vx, vy)
            (ctx.leapfrog_graph if graph else ctx.leapfrog)(3, 1e-2, 0.6)
        out.append(ctx.learned_export()[0])
        ctx.close()
    assert np.any(out[0]) and np.array_equal(out[0], out[1])


@pytest.mark.parametrize("n,near", [(300, 300), (900, 280), (1500, 1500)])
def test_refused_affinities_name_the_points(gpu, n, near):
    """Hundreds of near duplicates: refused, and the message counts each point with too many
    candidates once, whatever the number of column ranges (two for 1,500 points)."""
    rng = np.random.default_rng(n)
    X = rng.normal(0, 1, (n, 32))
    X[n - near:] = 5.0 + 1e-5 * rng.normal(0, 1, (near, 32))
    with pytest.raises(BHError) as e:
        tsne.affinities(X.astype(np.float32), perplexity=10.0, k=30)
    assert e.value.status == _lib.BH_ERR_CAPACITY
    assert f"{near} points have" in str(e.value)


@pytest.mark.parametrize("n", [50, 700])
@pytest.mark.parametrize("scale", [1e-38, 3e-42, 3e37])
def test_affinities_of_the_smallest_and_largest_inputs(gpu, n, scale):
    """Inputs whose scaling to FP16 takes a factor beyond a float's exponent (1e-38 and subnormal ones),
    and near the largest floats: the exact neighbours, distances to 1e-12."""
    rng = np.random.default_rng(n)
    k = 20
    X = (np.clip(rng.normal(0, 1, (n, 8)), -4, 4) * scale).astype(np.float32)
    assert np.all(np.isfinite(X))
    a = tsne.affinities(X, perplexity=6.0, k=k)
    d = X.astype(np.float64) / scale  # (the squares of 1e-42 in FP64 are exact enough; keep them near 1)
    d2 = ((d[:, None, :] - d[None, :, :]) ** 2).sum(2)
    np.fill_diagonal(d2, np.inf)
    want = np.sort(d2, axis=1)[:, :k]
    assert np.allclose(a["d2"] / scale / scale, want, rtol=1e-12, atol=0)
    got = np.take_along_axis(d2, a["idx"].astype(np.int64), 1)
    assert np.allclose(got, want, rtol=1e-12, atol=0)
    assert a["row_ptr"][n] == a["val"].size and np.all(a["col"] < n)
