"""Pair kernels that share one reciprocal among four denominators where that reciprocal is out of
range: the sums are those of a reciprocal each.  kernel_eps = 1e100 overflows every product of
four; kernel_eps = 0 makes the denominators of some coincident pairs exactly zero, which may spoil
the target they belong to and no other."""
import numpy as np
import pytest

from conftest import to_gpu, to_np

pytestmark = pytest.mark.gpu

# levels, proxy degree, leaf grid side: 16 waves per tile, lane copies of two rows, a row per lane
TREES = [(3, 6, 7), (5, 8, 6), (5, 8, 8)]


def make(sb, orc, p, eps):
    levels, d, m = p
    ctx = sb.Context(sb.RunConfig(levels=levels, interp_degree=d, leaf_degree=m - 1, kernel_eps=eps,
                                  weights="clenshaw_curtis"))
    return ctx, orc.OracleFMM(levels, d, m - 1, 0.7, 1)


@pytest.mark.parametrize("p", TREES, ids=lambda p: "L%d-d%d-m%d" % p)
def test_product_of_four_out_of_range(sb, orc, torch_gpu, p):
    """Both sides sum the same terms q / eps x cross y, so they agree to the rounding of the sums."""
    t, eps = torch_gpu, 1e100
    print(f"\n[case L{p[0]} d{p[1]} m{p[2]}]", flush=True)
    ctx, o = make(sb, orc, p, eps)
    x, y, z, a = o.spec_points()
    rng = np.random.default_rng(1)
    qp, qx = rng.normal(size=x.shape), rng.normal(size=(ctx.sizes.P, ctx.sizes.n))
    up = lambda *v: [to_gpu(t, w) for w in v]

    def close(got, expect):
        for g, e in zip(got, expect):
            g, e = to_np(g) * eps, np.asarray(e).reshape(x.shape) * eps
            assert np.all(np.isfinite(g)) and np.linalg.norm(g - e) <= 1e-12 * np.linalg.norm(e)

    close(ctx.bve_vel_interactions(*up(qp, qx))[0], o.bve_vel_interactions(qp, qx, eps, None, None)[0])
    rp, rx = np.roll(qp, 7), np.roll(qx, 7)
    for variant in (1, 2):
        close(ctx.swe_vel_interactions(*up(qp, qx, rp, rx), variant=variant)[0],
              o.swe_vel_interactions(variant, qp, qx, rp, rx, eps, None, None)[0])
    q, u = rng.normal(size=x.shape), [rng.normal(size=x.shape) for _ in range(3)]
    ga = to_gpu(t, a)
    v = [to_np(w) * eps for w in ctx.bve_velocity(ga, to_gpu(t, q))]
    qb = to_np(ctx.bve_velocity_adjoint(ga, up(*u))) * eps
    size = np.sqrt(sum(np.sum(w * w) for w in u) * sum(np.sum(w * w) for w in v))
    assert np.all(np.isfinite(qb))
    assert abs(sum(float(np.sum(b * w)) for b, w in zip(u, v)) - float(np.sum(qb * q))) <= 1e-12 * size
    # the direct sum from the particles at some of them
    pts = [w.ravel()[:300] for w in (x, y, z)]
    s = [w.ravel() for w in (x, y, z)]
    got = ctx.direct_sum_bve_vel_targets(*up(*pts), *up(*s), ga.reshape(-1), to_gpu(t, q.ravel()))
    f = (a * q).ravel() / (-4 * np.pi)
    sums = [float(np.sum(f * w)) for w in s]
    for c in range(3):
        i, j = (c + 1) % 3, (c + 2) % 3
        e = pts[i] * sums[j] - pts[j] * sums[i]
        assert np.linalg.norm(to_np(got[c]) * eps - e) <= 1e-12 * np.sqrt(300) * np.sum(np.abs(f))


def test_zero_denominator_stays_in_its_row(sb, orc, torch_gpu):
    """A lane holds rows i and 18 + i of a leaf's 36; coincident pairs with 1 - x.y exactly zero are
    met by some rows and not by others, so the two halves differ in which rows are finite."""
    t = torch_gpu
    ctx, o = make(sb, orc, (5, 8, 6), 0.0)
    x, _, _, a = o.spec_points()
    rng = np.random.default_rng(2)
    qp, qx = rng.normal(size=x.shape), rng.normal(size=(ctx.sizes.P, ctx.sizes.n))
    w = ctx.bve_vel_interactions(to_gpu(t, qp), to_gpu(t, qx))[0][0]
    s = ctx.swe_vel_interactions(*[to_gpu(t, v) for v in (qp, qx, qp, qx)])[0][0]
    b = ctx.bve_velocity_adjoint(to_gpu(t, a), [to_gpu(t, rng.normal(size=x.shape)) for _ in range(3)])
    for rows in (w, s, b):
        ok = np.isfinite(to_np(rows)).reshape(-1, 2, 18)
        assert np.any(ok[:, 0] != ok[:, 1])
