"""FP64 pair kernels whose workgroups share a target tile (csrc/pairwalk.hpp) against the
oracle: a row per lane at 16, 8 and 4 waves per tile, lane copies (csrc/lanes.hpp) at 8, 4 and 1,
source sets that batches of four, parts of a set and chunks of sets divide unevenly (9, 16, 25, 36,
49, 64, 81 and 121 points), one and two tiles per panel, accumulating and displaced.  Both sides sum the same pairs: 1e-12 leaves room for the rounding of 1 - x.y
(a few units of 1e-16 over eps = 1e-4) at the nearest pairs."""
import numpy as np
import pytest

from conftest import to_gpu, to_np

pytestmark = pytest.mark.gpu

EPS = 1e-4
# levels, proxy degree, leaf grid side: tile lists of 30 to 8,190; tiles of 9 and 16 rows, where a
# chunk of staged records spans several sets; more than 42 rows at 2,556 and 8,190 tiles
TREES = [(2, 4, 5), (3, 6, 7), (3, 8, 9), (4, 10, 11), (5, 8, 6), (6, 5, 6), (4, 2, 3), (5, 3, 4), (6, 2, 3),
         (5, 8, 8), (6, 6, 7)]


@pytest.fixture(scope="module", params=TREES, ids=lambda p: "L%d-d%d-m%d" % p)
def case(request, sb, orc, torch_gpu):
    levels, d, m = request.param
    print(f"\n[case L{levels} d{d} m{m}]", flush=True)
    ctx = sb.Context(sb.RunConfig(levels=levels, interp_degree=d, leaf_degree=m - 1, kernel_eps=EPS,
                                  weights="clenshaw_curtis"))
    o = orc.OracleFMM(levels, d, m - 1, 0.7, 1)
    x, y, z, a = o.spec_points()
    rng = np.random.default_rng(levels + d)
    qp, qx = rng.normal(size=x.shape), rng.normal(size=(ctx.sizes.P, ctx.sizes.n))
    dp = [1e-3 * rng.normal(size=x.shape) for _ in range(3)]
    dx = [1e-3 * rng.normal(size=qx.shape) for _ in range(3)]
    return dict(ctx=ctx, o=o, t=torch_gpu, W=sb.workloads, qp=qp, qx=qx, dp=dp, dx=dx, a=a, shape=x.shape)


def up(case, arrays):
    return [to_gpu(case["t"], v) for v in arrays]


def close(case, got_part, got_proxy, part, proxy, start=0.0):
    """Particle rows and the rows of non-leaf panels (leaf proxy rows are not targets)."""
    case["ctx"].synchronize()
    off = case["o"].offset
    for g, e in zip(got_part, part):
        e = np.asarray(e).reshape(case["shape"]) + start
        assert np.linalg.norm(to_np(g) - e) <= 1e-12 * np.linalg.norm(e)
    for g, e in zip(got_proxy, proxy):
        e = np.asarray(e)[:off] + start
        if np.any(np.asarray(e) != start):
            assert np.linalg.norm(to_np(g)[:off] - e) <= 1e-12 * np.linalg.norm(e)


@pytest.mark.parametrize("displaced", [False, True])
def test_vortex_pairs(case, displaced):
    ctx, o = case["ctx"], case["o"]
    dp, dx = (case["dp"], case["dx"]) if displaced else (None, None)
    ep, ex = o.bve_vel_interactions(case["qp"], case["qx"], EPS, dp, dx)
    phi_part, phi_proxy = ctx.zeros_part(3), ctx.zeros_proxy(3)
    for v in phi_part + phi_proxy:
        v.fill_(0.5)
    gp, gx = ctx.bve_vel_interactions(*up(case, [case["qp"], case["qx"]]), up(case, dp) if dp else None,
                                      up(case, dx) if dx else None, phi_part=phi_part, phi_proxy=phi_proxy)
    close(case, gp, gx, ep, ex, 0.5)


def test_log_pairs(case):
    """Coincident nodes (a tile's own leaf, shared leaf edges) are skipped on both sides."""
    ctx, o = case["ctx"], case["o"]
    ep, ex = o.poisson_fmm_interactions(case["qp"], case["qx"])
    psi_part, psi_proxy = ctx.zeros_part(), ctx.zeros_proxy()
    for v in (psi_part, psi_proxy):
        v.fill_(0.5)
    gp, gx = ctx.poisson_fmm_interactions(*up(case, [case["qp"], case["qx"]]), psi_part, psi_proxy)
    close(case, [gp], [gx], [ep], [ex], 0.5)


@pytest.mark.parametrize("variant", [1, 2])
@pytest.mark.parametrize("displaced", [False, True])
def test_shallow_water_pairs(case, variant, displaced):
    ctx, o = case["ctx"], case["o"]
    dp, dx = (case["dp"], case["dx"]) if displaced else (None, None)
    dpart, dprox = np.roll(case["qp"], 7), np.roll(case["qx"], 7)
    ep, ex = o.swe_vel_interactions(variant, case["qp"], case["qx"], dpart, dprox, EPS, dp, dx)
    phi_part, phi_proxy = ctx.zeros_part(3), ctx.zeros_proxy(3)
    for v in phi_part + phi_proxy:
        v.fill_(0.5)
    gp, gx = ctx.swe_vel_interactions(*up(case, [case["qp"], case["qx"], dpart, dprox]), up(case, dp) if dp else None,
                                      up(case, dx) if dx else None, phi_part, phi_proxy, variant)
    close(case, gp, gx, ep, ex, 0.5)


@pytest.mark.parametrize("displaced", [False, True])
def test_laplacian_pairs(case, displaced):
    ctx, o = case["ctx"], case["o"]
    dp, dx = (case["dp"], case["dx"]) if displaced else (None, None)
    ep, ex = o.laplacian_interactions(case["qp"], case["qx"], dp, dx)
    phi_part, phi_proxy = ctx.zeros_part(), ctx.zeros_proxy()
    for v in (phi_part, phi_proxy):
        v.fill_(0.5)
    gp, gx = ctx.laplacian_interactions(*up(case, [case["qp"], case["qx"]]), up(case, dp) if dp else None,
                                        up(case, dx) if dx else None, phi_part, phi_proxy)
    close(case, [gp], [gx], [ep], [ex], 0.5)


@pytest.mark.parametrize("displaced", [False, True])
def test_vortex_pairs_mixed(case, displaced, sb):
    """Lane copies of 13 to 32 lanes (tiles of 25 to 64 targets), chunks and sets that they divide
    unevenly.  In panel-centred FP32 the denominator alpha + beta - p.b is off by a few 2^-24 of
    r^2 (r the leaf radius), which the nearest pairs (eps) magnify, on top of a few 2^-24 per pair;
    the per-pair bound 2^-24 (8 + 2 r^2 / eps) bounds the field's relative error."""
    ctx, o, W = case["ctx"], case["o"], case["W"]
    cm = sb.Context(sb.RunConfig(levels=ctx.cfg.levels, interp_degree=ctx.cfg.interp_degree,
                                 leaf_degree=ctx.cfg.leaf_degree, kernel_eps=EPS, weights="clenshaw_curtis",
                                 precision="mixed"))
    x, y, z, a = o.spec_points()
    qp, qx = o.upward_pass(a, W.gaussian_vortices(x, y, z, a, seed=3))
    dp, dx = (case["dp"], case["dx"]) if displaced else (None, None)
    ep, ex = o.bve_vel_interactions(qp, qx, EPS, dp, dx)
    gp, gx = cm.bve_vel_interactions(*up(case, [qp, qx]), up(case, dp) if dp else None, up(case, dx) if dx else None)
    cm.synchronize()
    r = np.sqrt(2) * (np.pi / 4) / 2 ** (ctx.cfg.levels - 1)
    bound = 2.0 ** -24 * (8 + 2 * r * r / EPS)
    assert W.vec_rel_l2([to_np(v) for v in gp], ep) < bound
    off = o.offset
    if np.any([np.any(np.asarray(v)[:off]) for v in ex]):
        assert W.vec_rel_l2([to_np(v)[:off] for v in gx], [np.asarray(v)[:off] for v in ex]) < bound


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_velocity_adjoint_is_the_transpose(case, precision, sb):
    """<u, K q> = <K^T u, q>: both sides sum the same pairs, so they agree to the rounding of the
    pair sums (FP64 as above; the FP32 bound of test_vortex_pairs_mixed) times the operands' norms."""
    cfg = case["ctx"].cfg
    ctx = sb.Context(sb.RunConfig(levels=cfg.levels, interp_degree=cfg.interp_degree, leaf_degree=cfg.leaf_degree,
                                  kernel_eps=EPS, weights="clenshaw_curtis", precision=precision))
    x, y, z, a = case["o"].spec_points()
    rng = np.random.default_rng(4)
    q, u = rng.normal(size=x.shape), [rng.normal(size=x.shape) for _ in range(3)]
    ga = to_gpu(case["t"], a)
    v = [to_np(w) for w in ctx.bve_velocity(ga, to_gpu(case["t"], q))]
    qb = to_np(ctx.bve_velocity_adjoint(ga, up(case, u)))
    lhs, rhs = sum(float(np.sum(p * w)) for p, w in zip(u, v)), float(np.sum(qb * q))
    size = np.sqrt(sum(np.sum(p * p) for p in u) * sum(np.sum(w * w) for w in v))
    r = np.sqrt(2) * (np.pi / 4) / 2 ** (cfg.levels - 1)
    assert abs(lhs - rhs) <= (1e-12 if precision == "fp64" else 2.0 ** -24 * (8 + 2 * r * r / EPS)) * size


@pytest.mark.parametrize("displaced", [False, True])
def test_other_pairs_mixed(case, displaced, sb):
    """The FP32 shallow-water, regularised-Laplacian and log pairs in lane copies against the FP64
    kernels (above against the oracle).  Per pair: the shallow-water bound of
    test_vortex_pairs_mixed; the Laplacian's base-2 exponent, up to 2 / (0.1 ln 2) = 29, is off by
    half an ulp of itself, under 64 x 2^-24 with its polynomials; the logarithm by an ulp of up to
    -16 and 2 r^2 2^-24 over the nearest squared distance, of pairs that count as 1/N."""
    cfg, W = case["ctx"].cfg, case["W"]
    kw = dict(levels=cfg.levels, interp_degree=cfg.interp_degree, leaf_degree=cfg.leaf_degree, kernel_eps=EPS,
              weights="clenshaw_curtis")
    c64, c32 = case["ctx"], sb.Context(sb.RunConfig(precision="mixed", **kw))
    x, y, z, a = case["o"].spec_points()
    q = up(case, case["o"].upward_pass(a, W.gaussian_vortices(x, y, z, a, seed=3)))
    p = up(case, case["o"].upward_pass(a, W.gaussian_vortices(x, y, z, a, seed=4)))
    dp, dx = (up(case, case["dp"]), up(case, case["dx"])) if displaced else (None, None)
    r = np.sqrt(2) * (np.pi / 4) / 2 ** (cfg.levels - 1)
    off = case["o"].offset
    calls = [(lambda c: c.swe_vel_interactions(*q, *p, dp, dx), 8 + 2 * r * r / EPS),
             (lambda c: c.laplacian_interactions(*q, dp, dx), 64)]
    if not displaced:
        calls.append((lambda c: c.poisson_fmm_interactions(*q), 64))
    for call, bound in calls:
        (ep, ex), (gp, gx) = call(c64), call(c32)
        flat = lambda part, proxy: np.concatenate([to_np(v).ravel() for v in (part if isinstance(part, list) else [part])]
                                                  + [to_np(v)[:off].ravel() for v in
                                                     (proxy if isinstance(proxy, list) else [proxy])])
        e, g = flat(ep, ex), flat(gp, gx)
        assert np.linalg.norm(g - e) <= 2.0 ** -24 * bound * np.linalg.norm(e)


def test_step_adjoint_mixed_against_fp64(case, sb):
    """The step's gradient, whose displaced stages also take the position cotangents: two sets of
    kernels for the same sums.  A pair's g is off by the FP32 bound of test_vortex_pairs_mixed and
    its g^2 by twice that; the rest of the step is FP64 on both sides."""
    cfg, W = case["ctx"].cfg, case["W"]
    x, y, z, a = case["o"].spec_points()
    vor = W.gaussian_vortices(x, y, z, a, seed=3)
    bar = np.random.default_rng(5).normal(size=x.shape)
    got = []
    for precision in ("fp64", "mixed"):
        ctx = sb.Context(sb.RunConfig(levels=cfg.levels, interp_degree=cfg.interp_degree, leaf_degree=cfg.leaf_degree,
                                      kernel_eps=EPS, weights="clenshaw_curtis", precision=precision, delta_t=900.0))
        got.append(to_np(ctx.bve_back_rk4_step_adjoint(*up(case, [x, y, z, a, vor, bar]))))
        ctx.synchronize()
    r = np.sqrt(2) * (np.pi / 4) / 2 ** (cfg.levels - 1)
    err = np.linalg.norm(got[1] - got[0]) / np.linalg.norm(got[0])
    print(f"  step adjoint, mixed from fp64: {err:.2e}")
    assert err <= 3 * 2.0 ** -24 * (8 + 2 * r * r / EPS)
