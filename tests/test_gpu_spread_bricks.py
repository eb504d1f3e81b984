"""The double-layer spread by 4^3 bricks at its edges: grids that 4 does not divide, a grid of
barely a stencil and a brick, one below that (the general kernel), B-spline orders 4, 6 and 8,
cells outside the box; both layers and the double layer alone, against the oracle's grids and
velocities to 1e-12 (FP64 sums in another order), and the FP32 form to 1e-6."""
import numpy as np
import pytest

from oracle import oracle_py as O
from rbc3d_amd import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Nb,P", [((10, 30, 27), 6), ((9, 16, 18), 6), ((25, 18, 30), 4), ((12, 15, 20), 8),
                                  ((32, 32, 32), 6)])
def test_grids(Nb, P):
    import rbc3d_amd as R
    rng = np.random.default_rng(P)
    L = 8.0
    cs = configs.place_centres(rng, 3, (L, L, L), 2.2)
    cs[1] -= 2 * L
    cells = configs.build_cells(rng, ["disc"] * 3, [9, 12, 9], [1.0] * 3, cs, [1, 1, 1])
    w = configs.Workload("spread", (L, L, L), configs.alpha_ref_from_xi(1.5), 2.0, Nb, P, (5.0,),
                         (0.0, 0.0, 0.0), cells)
    g, o = R.from_workload(w), O.from_workload(w)
    tl = o.tlist_rbc()
    for c1, c2 in ((0.0, 0.7), (0.3, -0.7)):
        vo = o.pme(c1, c2, tl)
        for prec, tol in ((g.PREC_FP64, 1e-12), (g.PREC_SPLIT, 1e-6)):
            g.set_precision(prec)
            vg = g.pme(c1, c2, tl)
            for which in (0, 1) if c1 else (1,):
                a, b = g.pme_grid(which), o.pme_grid(which)
                assert np.abs(a - b).max() <= tol * np.abs(b).max(), (which, prec)
            err = np.abs(vg - vo).max() / np.abs(vo).max()
            assert err < tol, (c1, prec, err)
    print(f"grid {Nb}, order {P}: velocity {err:.2e}", flush=True)
