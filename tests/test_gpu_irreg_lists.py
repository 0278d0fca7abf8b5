"""Pair sums of irregular trees at the tile counts where their launch changes (below 400, 1,000
and 1,500, above 6,000), against the oracle and, on the largest, against each other.  Both sides
sum the same pairs: 1e-12 as in test_gpu_irreg.py."""
import numpy as np
import pytest

from conftest import to_gpu, to_np

pytestmark = pytest.mark.gpu

EPS = 1e-4
# points, points a leaf, degree
LISTS = [(2000, 40, 4), (4000, 20, 3), (9000, 30, 5), (20000, 12, 4)]


@pytest.mark.parametrize("n,leaf,degree", LISTS)
def test_irregular_lists(sb, orc, torch_gpu, n, leaf, degree):
    t = torch_gpu
    rng = np.random.default_rng(n)
    X = rng.normal(size=(3, n))
    X /= np.linalg.norm(X, axis=0)
    ctx = sb.Context(sb.RunConfig(levels=2, interp_degree=degree, kernel_eps=EPS))
    irr = ctx.irregular(*X, leaf)
    print(f"\n[case irregular N={n} leaf={leaf} d={degree}: {irr.tiles} tiles]", flush=True)
    area = np.full(n, 4 * np.pi / n) * (1 + 0.1 * rng.random(n))
    vor, div = X[2] + 0.3 * X[0] * X[1], 0.5 * X[0] - 0.2 * X[1] * X[2]
    ga, gv, gd = [to_gpu(t, v) for v in (area, vor, div)]
    swe = np.stack([to_np(v) for v in irr.swe_velocity(ga, gv, gd)], 1)
    zero = np.stack([to_np(v) for v in irr.swe_velocity(ga, gv, t.zeros_like(gv))], 1)
    bve = np.stack([to_np(v) for v in irr.bve_velocity(ga, gv)], 1)
    np.testing.assert_allclose(bve, zero, rtol=0, atol=1e-12 * np.abs(zero).max())
    if n <= 9000:
        ref = np.stack(orc.OracleIrreg(*X, leaf, degree, 0.7).swe_velocity(area, vor, div, EPS), 1)
        np.testing.assert_allclose(swe, ref, rtol=0, atol=1e-12 * np.abs(ref).max())
