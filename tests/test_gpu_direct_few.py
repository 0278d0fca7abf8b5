"""Direct sums of a few sources at more targets than fill the chip (a wave per target tile) against
numpy in FP64, at the edges of the rule: 1 and 128 sources, tile counts either side of 1,500 and of
25 per source, with remainders of a tile, and 129 sources, where waves always share a tile."""
import numpy as np
import pytest

from conftest import to_gpu, to_np

pytestmark = pytest.mark.gpu

EPS = 1e-4
U = 2.0 ** -53


@pytest.mark.parametrize("nt,ns", [(192000, 1), (191800, 5), (1400003, 3), (409600, 128), (409400, 128), (500001, 129)])
def test_few_sources(sb, torch_gpu, nt, ns):
    t, W = torch_gpu, sb.workloads
    print(f"\n[direct sums {nt} x {ns}]", flush=True)
    ctx = sb.Context(sb.RunConfig(levels=2, interp_degree=4, leaf_degree=4, kernel_eps=EPS))
    rng = np.random.default_rng(ns)
    src, tgt = W.random_unit_vectors(ns, seed=1), W.random_unit_vectors(nt, seed=2)
    for i, j in ((0, 0), (nt - 1, ns - 1)):  # targets on sources: guarded
        for k in range(3):
            tgt[k][i] = src[k][j]
    q, area = rng.normal(size=ns), np.full(ns, 1.0 / ns)
    g = lambda v: [to_gpu(t, w) for w in v]
    ga, gq = to_gpu(t, area), to_gpu(t, q)
    psi = to_np(ctx.direct_sum_inv_lap_targets(*g(tgt), *g(src), ga, gq))
    vel = [to_np(v) for v in ctx.direct_sum_bve_vel_targets(*g(tgt), *g(src), ga, gq)]
    f, w = area * q, np.abs(area * q)
    ref, size = np.zeros(nt), np.zeros(nt)
    s, size_v = np.zeros((3, nt)), np.zeros((3, nt))
    # the bounds of test_gpu_direct_shapes.py, source by source; near x.y = 0, where a single logarithm
    # is small, the table's error is absolute (2^-58)
    for j in range(ns):
        d = 1.0 - (tgt[0] * src[0][j] + tgt[1] * src[1][j] + tgt[2] * src[2][j])
        term = np.where(1.0 - d < 1.0 - 1e-15, np.log(np.maximum(d, 1e-300)), 0.0)
        ref -= term * f[j] / (4 * np.pi)
        size += ((ns + 8) * U * np.abs(term) + 2.0 ** -57) * w[j]
        d += EPS
        for c in range(3):
            a, b = (c + 1) % 3, (c + 2) % 3
            s[c] -= (tgt[a] * src[b][j] - tgt[b] * src[a][j]) / d * f[j] / (4 * np.pi)
            size_v[c] += ((ns + 12) * U + 8 * U / d) * (np.abs(tgt[a] * src[b][j]) + np.abs(tgt[b] * src[a][j])) / d * w[j]
    assert np.all(np.abs(psi - ref) <= size)
    for c in range(3):
        assert np.all(np.abs(vel[c] - s[c]) <= size_v[c])
