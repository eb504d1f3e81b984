"""Neighbouring-cell lists: the number of (target, cell) pairs within the cut-off against a
brute-force count, and the matvec that follows from the closest nodes against the oracle to
1e-12; boxes that cells wrap around and not, grids of 2 to 32 latitudes, cells on a lattice
whose closest nodes come in ties."""
import numpy as np
import pytest

from oracle import oracle_py as O
from rbc3d_amd import configs

pytestmark = pytest.mark.gpu

CASES = {
    "wide": ((12.0,) * 3, 2.0, 12, (13,), False),
    "wrapped": ((5.0, 5.3, 6.0), 1.7, 3, (9, 13), False),
    "one_bin": ((4.6, 9.0, 4.6), 2.2, 3, (6,), False),
    "fine_and_coarse": ((8.0,) * 3, 1.9, 6, (24, 2, 32, 9), False),
    "lattice": ((7.5,) * 3, 2.5, 27, (6,), True),
}


@pytest.mark.parametrize("name", CASES)
def test_lists(name):
    import rbc3d_amd as R
    Lb, rc, n, nlats, lattice = CASES[name]
    rng = np.random.default_rng(len(name))
    if lattice:
        k = round(n ** (1 / 3))
        g1 = (np.arange(k) + 0.5) * Lb[0] / k
        cs = np.stack(np.meshgrid(g1, g1, g1, indexing="ij"), -1).reshape(-1, 3)
    else:
        cs = configs.place_centres(rng, n, Lb, 2.1 if n > 3 else 2.0)
    nl = [nlats[k % len(nlats)] for k in range(n)]
    kind = "sphere" if lattice else "disc"
    cells = configs.build_cells(rng, [kind] * n, nl, [1.0] * n, cs, [1] * n,
                                rots=[np.eye(3)] * n if lattice else None)
    w = configs.Workload(name, Lb, configs.alpha_ref_from_xi(2.0), rc, (32,) * 3, 6,
                         (5.0, 1.0), (0.0, 0.0, 0.0), cells)
    g, o = R.from_workload(w), O.from_workload(w)
    u = rng.standard_normal(g.cell_dof())
    bg, bo = g.cell_matmult(u), o.cell_matmult(u)
    ends = np.cumsum([6 * m * m for m in nl])
    xs = [cells.x[e - 6 * m * m:e].reshape(-1, 3, order="F") for e, m in zip(ends, nl)]
    L = np.asarray(Lb)
    count = 0
    for i, xi in enumerate(xs):
        for j, xj in enumerate(xs):
            if i != j:
                d = xi[:, None] - xj[None]
                d -= np.round(d / L) * L
                count += int(((d ** 2).sum(-1).min(1) <= rc * rc).sum())
    err = np.abs(bg - bo).max() / np.abs(bo).max()
    print(f"{name}: {count} lists, {g.near_stats()}, matvec {err:.2e}", flush=True)
    assert g.near_stats()[0] == count
    assert err < 1e-12
