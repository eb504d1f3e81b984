"""The pair kernels' target clusters at their edges: target counts around the cluster size,
inactive targets, targets and sources outside the periodic box, boxes small enough for the
minimum-image formula and large enough for the bin walk's images.  AddIntOnRbcs against the
oracle: pair set exact, velocities to 1e-12 (FP64 sums in another order)."""
import numpy as np
import pytest

from oracle import oracle_py as O
from rbc3d_amd import configs

pytestmark = pytest.mark.gpu
TOL = 1e-12


def suspension(L, ncell, seed, shift):
    """Discs of two viscosity ratios (one of them 1); with `shift` every third cell lies a
    period or two outside the box."""
    rng = np.random.default_rng(seed)
    cs = configs.place_centres(rng, ncell, (L, L, L), 2.2)
    if shift:
        cs[::3] += L * np.array([1.0, -2.0, 1.0])
    types = [1 + (k % 2) for k in range(ncell)]
    cells = configs.build_cells(rng, ["disc"] * ncell, [11] * ncell, [1.0] * ncell, cs, types)
    return configs.Workload("pairs", (L, L, L), configs.alpha_ref_from_xi(2.0), 2.0, (32,) * 3, 6,
                            (5.0, 1.0), (0.0, 0.0, 0.0), cells)


@pytest.mark.parametrize("L,ncell,shift", [(8.0, 4, False), (8.0, 4, True), (13.0, 24, True)])
def test_clusters(L, ncell, shift):
    import rbc3d_amd as R
    w = suspension(L, ncell, 7, shift)
    g, o = R.from_workload(w), O.from_workload(w)
    rng = np.random.default_rng(3)
    c = 1 / (4 * np.pi)
    tx, ti, act, A = o.tlist_rbc()
    n = len(A)
    lists = [(tx, ti, act, A), (tx, ti, (rng.random(n) < 0.4).astype(np.int32), A)]
    for m in (1, 7, 8, 9, 65):  # free points, some of them outside the box
        x = rng.uniform(-1.5 * L, 2.5 * L, 3 * m)
        lists.append((x, np.zeros(3 * m, np.int32), np.ones(m, np.int32), rng.uniform(1, 2, m)))
    for tl in lists:
        for c1, c2 in ((0.0, -c), (c, 0.0), (c, -c)):
            vo, npairs = o.add_int_on_rbcs(c1, c2, tl)
            vg = g.add_int_on_rbcs(c1, c2, tl)
            ng, cs = g.pair_stats()
            assert ng == npairs and cs == o.pair_checksum(), (len(tl[3]), c1, c2)
            err = np.abs(vg - vo).max() / np.abs(vo).max()
            assert err < TOL, (len(tl[3]), c1, c2, err)
    print(f"box {L}: {ng} pairs in the last list", flush=True)


def test_viscosity_ratio_one():
    """Cells without a double layer (Bcoef = 0): the double-layer pair sums vanish."""
    import rbc3d_amd as R
    w = suspension(13.0, 6, 9, False)
    w.viscRat = (1.0, 1.0)
    g, o = R.from_workload(w), O.from_workload(w)
    tl = o.tlist_rbc()
    for c1, c2 in ((0.5, -0.5), (0.0, -0.5)):
        vo, npairs = o.add_int_on_rbcs(c1, c2, tl)
        vg = g.add_int_on_rbcs(c1, c2, tl)
        assert g.pair_stats()[0] == npairs
        assert np.abs(vg - vo).max() <= TOL * max(np.abs(vo).max(), 1.0)


@pytest.mark.parametrize("L", [13.0, 5.0])
def test_far_targets(L):
    """Points so many periods away that their bins' numbers leave 32 bits, in one cluster with
    points in the box: these keep their velocities."""
    import rbc3d_amd as R
    w = suspension(L, 6 if L > 8 else 1, 11, False)
    g, o = R.from_workload(w), O.from_workload(w)
    rng = np.random.default_rng(2)
    Nf = 2 * max(int(L // w.rc), 3)
    bins = np.array([(2**31 - 1) % Nf, (-2**31) % Nf])  # the bins that such points fall in
    near = ((bins[:, None, None] + rng.random((2, 7, 3))) * L / Nf).reshape(-1, 3)
    pts = np.concatenate([near, [[1e13] * 3, [-1e13] * 3]])

    def tl(p):
        k = len(p)
        return p.reshape(-1, order="F").copy(), np.zeros(3 * k, np.int32), np.ones(k, np.int32), np.ones(k)

    for c1, c2 in ((0.0, 1.0), (0.7, -1.3)):
        vo = o.add_int_on_rbcs(c1, c2, tl(near))[0].reshape(3, -1)
        vg = g.add_int_on_rbcs(c1, c2, tl(pts)).reshape(3, -1)[:, :len(near)]
        assert np.abs(vo).max() > 0
        err = np.abs(vg - vo).max() / np.abs(vo).max()
        print(f"box {L}, {c1}, {c2}: {err:.2e}", flush=True)
        assert err < TOL


def test_undefined_other_density():
    """A layer that a sum leaves out does not enter it: the single layer's density undefined, the
    double layer summed, with and without cells that carry one."""
    import rbc3d_amd as R
    for ratios in ((1.0, 1.0), (5.0, 1.0)):
        w = suspension(13.0, 24, 7, False)
        w.viscRat = ratios
        g, o = R.from_workload(w), O.from_workload(w)
        tl = o.tlist_rbc()
        vo, _ = o.add_int_on_rbcs(0.0, 0.7, tl)
        g.set_cell_density(1, np.full_like(w.cells.f, np.nan))
        vg = g.add_int_on_rbcs(0.0, 0.7, tl)
        assert g.near_stats()[1] > 0
        assert np.abs(vg - vo).max() <= TOL * max(np.abs(vo).max(), 1.0), ratios
