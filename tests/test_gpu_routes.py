"""Calls whose path depends on their size or input, on each path that the other tests leave out: the
learned walk with one, two and four waves per group and with totals."""
import numpy as np
import pytest

from masterthesislucas_amd.learned import N_OUT, FarFieldMLP, flatten
from oracle import oracle as O
from tests.helpers import WALK_TOL, exact_walk
from tests.test_gpu_learned import _gpu_tree, _params, _plummer_ctx

pytestmark = pytest.mark.gpu

EPS = float(np.float32(1e-3))


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
