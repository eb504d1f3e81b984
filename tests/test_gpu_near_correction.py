"""The near-singular correction of either layer and of both, at points from half a mesh width
down to 0.002 of it, inside and outside (on the surface itself the jump's side is rounding),
poles included; grids of 6 to 40 latitudes, cells with and without a double layer.  Against the
oracle.  The tolerance is measured from the problem: coordinates moved by two units in the last
place change the oracle's own result by some amount (most on 6 latitudes, whose closest points
three fit steps leave unconverged), and the kernel, which rounds about 10 such coordinate-sized
operations between a point and its result, may differ by 16 times that, and 1e-12 in sums."""
import numpy as np
import pytest

from oracle import oracle_py as O
from rbc3d_amd import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nlats", [(6, 13), (24, 9), (32,), (40,)])
@pytest.mark.parametrize("c1,c2", [(1.0, 0.0), (0.0, 1.0), (0.7, -1.3)])
def test_points_near_cells(nlats, c1, c2):
    import rbc3d_amd as R
    rng = np.random.default_rng(sum(nlats))
    n, L = 2, 8.0
    cs = configs.place_centres(rng, n, (L, L, L), 2.4)
    nl = [nlats[k % len(nlats)] for k in range(n)]
    cells = configs.build_cells(rng, ["disc"] * n, nl, [1.0] * n, cs, [1, 2])
    w = configs.Workload("near", (L,) * 3, configs.alpha_ref_from_xi(2.0), 2.0, (32,) * 3, 6,
                         (5.0, 1.0), (0.0, 0.0, 0.0), cells)
    g, o = R.from_workload(w), O.from_workload(w)
    pts, off = [], 0
    for m in nl:
        x = cells.x[off:off + 6 * m * m].reshape(-1, 3, order="F")
        a3 = cells.a3[off:off + 6 * m * m].reshape(-1, 3, order="F")
        off += 6 * m * m
        q = np.concatenate([[0, m - 1, m // 2], rng.integers(0, 2 * m * m, 13)])
        for h in (0.5, -0.5, 0.05, -0.05, 0.002, -0.002):
            pts.append(x[q] + h * 3.5 / m * a3[q] + (0.2 / m) * rng.standard_normal((16, 3)) * (h == 0.5))
    x = np.concatenate(pts)
    k = len(x)
    tl = (x.reshape(-1, order="F").copy(), np.zeros(k, np.int32), np.ones(k, np.int32), np.ones(k))
    vo, _ = o.add_int_on_rbcs(c1, c2, tl)
    top, sens = np.abs(vo).max(), 0.0
    for _ in range(4):
        moved = tl[0] * (1 + 2.0**-51 * rng.choice([-1.0, 1.0], tl[0].shape))
        sens = max(sens, np.abs(o.add_int_on_rbcs(c1, c2, (moved, *tl[1:]))[0] - vo).max() / top)
    vg = g.add_int_on_rbcs(c1, c2, tl)
    err = np.abs(vg - vo).max() / top
    print(f"grids {nlats}, c {c1}, {c2}: {g.near_stats()}, {err:.2e}, sensitivity {sens:.2e}", flush=True)
    assert g.near_stats()[1] >= k
    assert err < 1e-12 + 16 * sens
    # the sensitivities measured: up to 4.0e-12 on 6 latitudes' double layer, 7.9e-14 elsewhere
    assert sens < (1e-11 if c2 != 0 and min(nlats) == 6 else 2e-13)
