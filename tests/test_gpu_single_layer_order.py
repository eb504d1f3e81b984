"""The single layer's sums and near-singular corrections bit for bit as recorded
(tests/golden/single_layer_near.npz: 192 points near two discs of 6 and 9 latitudes, all
corrected, down to 0.0007 from the surface).  Wall solves follow the last bits of these sums, so
their order and contractions are fixed in the kernels; a new record is due only where the
device or host library's own functions change.  Against the oracle the values hold to 1e-12."""
import os

import numpy as np
import pytest

from oracle import oracle_py as O
from rbc3d_amd import configs

pytestmark = pytest.mark.gpu
RECORD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "single_layer_near.npz")


def test_recorded_bits():
    import rbc3d_amd as R
    z = np.load(RECORD)
    nl, L = z["nlat"], 8.0
    cells = configs.Cells(nlat0=nl, nlat=nl, celltype=np.ones(len(nl), np.int32), x=z["x"], a3=z["a3"],
                          detj=z["detj"], f=z["f"], g=z["g"])
    w = configs.Workload("near", (L,) * 3, configs.alpha_ref_from_xi(2.0), 2.0, (32,) * 3, 6, (1.0,),
                         (0.0, 0.0, 0.0), cells)
    g, o = R.from_workload(w), O.from_workload(w)
    k = len(z["points"]) // 3
    tl = (z["points"], np.zeros(3 * k, np.int32), np.ones(k, np.int32), np.ones(k))
    v = g.add_int_on_rbcs(1.0, 0.0, tl)
    assert g.near_stats() == (193, 192)
    vo = o.add_int_on_rbcs(1.0, 0.0, tl)[0]
    err = np.abs(v - vo).max() / np.abs(vo).max()
    print(f"{k} points: {(v != z['velocity']).sum()} values differ from the record, oracle {err:.2e}", flush=True)
    assert err < 1e-12
    assert np.array_equal(v, z["velocity"])
