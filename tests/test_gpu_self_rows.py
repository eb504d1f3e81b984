"""The self patch by latitude rows (cell matvec): enough cells to take that path, grids whose
spline band fits the LDS and one whose does not, against the oracle to 1e-12."""
import numpy as np
import pytest

from oracle import oracle_py as O
from rbc3d_amd import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nlats", [(6,), (9, 12), (13,), (17, 11), (24,)])
def test_rows(nlats):
    import rbc3d_amd as R
    rng = np.random.default_rng(sum(nlats))
    n, L = 22 if max(nlats) < 20 else 8, 12.0
    cs = configs.place_centres(rng, n, (L, L, L), 2.3)
    nl = [nlats[k % len(nlats)] for k in range(n)]
    cells = configs.build_cells(rng, ["disc"] * n, nl, [1.0] * n, cs, [1 + k % 2 for k in range(n)])
    w = configs.Workload("rows", (L, L, L), configs.alpha_ref_from_xi(2.0), 2.0, (32,) * 3, 6,
                         (5.0, 1.0), (0.0, 0.0, 0.0), cells)
    import torch
    # enough rows for this device to take the path
    assert 2 * sum(nl) >= torch.cuda.get_device_properties(0).multi_processor_count
    g, o = R.from_workload(w), O.from_workload(w)
    u = rng.standard_normal(g.cell_dof())
    bg, bo = g.cell_matmult(u), o.cell_matmult(u)
    err = np.abs(bg - bo).max() / np.abs(bo).max()
    print(f"grids {nlats}: {sum(nl)} rows, matvec {err:.2e}", flush=True)
    assert err < 1e-12
