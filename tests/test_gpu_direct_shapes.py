"""Direct sums at the edges of their tiling (64 or 128 targets per workgroup, eight waves
sharing a source chunk, batches of four sources) against numpy in FP64, with the guarded
pairs (a target's own source, coincident points) in first, last and inner batches."""
import numpy as np
import pytest

from conftest import to_gpu, to_np

pytestmark = pytest.mark.gpu

EPS = 1e-4
U = 2.0 ** -53
# targets x sources: one pair; batch and wave remainders; one, two, odd and many 64-target rows;
# one and several 256-source chunks
SHAPES = [(1, 1), (3, 5), (64, 255), (65, 256), (128, 259), (192, 1027), (575, 513), (513, 2049)]


def dots(t, s):
    return t[0][:, None] * s[0] + t[1][:, None] * s[1] + t[2][:, None] * s[2]


@pytest.fixture(scope="module")
def ctx(sb, torch_gpu):
    return sb.Context(sb.RunConfig(levels=2, interp_degree=4, leaf_degree=4, kernel_eps=EPS))


@pytest.mark.parametrize("nt,ns", SHAPES)
def test_direct_sums_at_tile_edges(sb, torch_gpu, ctx, nt, ns):
    t, W = torch_gpu, sb.workloads
    print(f"\n[direct sums {nt} x {ns}]", flush=True)
    rng = np.random.default_rng(nt + ns)
    src, tgt = W.random_unit_vectors(ns, seed=1), W.random_unit_vectors(nt, seed=2)
    for i, j in ((0, 0), (nt - 1, ns - 1), (nt // 2, ns // 2)):  # targets on sources: guarded
        for k in range(3):
            tgt[k][i] = src[k][j]
    area, q = rng.uniform(0.5, 1.5, ns) / ns, rng.normal(size=ns)
    gs, gt = [to_gpu(t, v) for v in src], [to_gpu(t, v) for v in tgt]
    ga, gq = to_gpu(t, area), to_gpu(t, q)
    w = np.abs(area * q)

    # log sum at separate targets, coincident pairs skipped.  Per pair: both logarithms within
    # 1.2 ulp, the same x.y on both sides; then ns additions of either side.
    dp = dots(tgt, src)
    skip = ~(dp < 1.0 - 1e-15)
    term = np.where(skip, 0.0, np.log(np.maximum(1.0 - dp, 1e-300)))
    got = to_np(ctx.direct_sum_inv_lap_targets(*gt, *gs, ga, gq))
    assert np.all(np.abs(got + (term @ (area * q)) / (4 * np.pi)) <= (ns + 8) * U * (np.abs(term) @ w))

    # log sum over the points themselves, i != j, on a slice
    lb, ub = ns // 5, ns - ns // 7
    dp = dots(src, src)
    term = np.log(np.maximum(1.0 - dp, 1e-300))
    np.fill_diagonal(term, 0.0)
    got = to_np(ctx.direct_sum_inv_lap(*gs, ga, gq, lb=lb, ub=ub))
    expect = -(term @ (area * q)) / (4 * np.pi)
    assert np.all(got[:lb] == 0) and np.all(got[ub:] == 0)
    assert np.all(np.abs(got - expect)[lb:ub] <= (ns + 8) * U * (np.abs(term) @ w)[lb:ub])

    # Biot-Savart: 1 - x.y is off by a few U on either side, which its reciprocal magnifies
    d = (1.0 - dots(tgt, src)) + EPS
    vel = ctx.direct_sum_bve_vel_targets(*gt, *gs, ga, gq)
    rel = (ns + 12) * U + 8 * U / d
    for c in range(3):
        a, b = (c + 1) % 3, (c + 2) % 3
        # the target multiplies the sum of g y, so either product counts, not their difference
        size = (np.abs(tgt[a])[:, None] * np.abs(src[b]) + np.abs(tgt[b])[:, None] * np.abs(src[a])) / d
        k = (tgt[a][:, None] * src[b] - tgt[b][:, None] * src[a]) / d
        expect = -(k @ (area * q)) / (4 * np.pi)
        assert np.all(np.abs(to_np(vel[c]) - expect) <= (size * rel) @ w)
