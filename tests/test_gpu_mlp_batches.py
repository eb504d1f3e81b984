"""The network's training kernel at the edges of its split (tiles of 16 nodes, up to four
wavefronts a workgroup, at most 256 workgroups) and its GELU far from zero, against the
CPU oracle."""
import numpy as np
import pytest

from oracle import mlp_oracle as M
from tests.test_gpu_mlp import _data, _net

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 16, 17, 64, 65, 4096, 4097, 8193, 16384, 16401])
def test_gradient_batches(n):
    import torch
    import rbc3d_amd as R
    m, p = _net(R, 5)
    X, T = _data(n, n)
    mean, std = np.zeros(9, np.float32), np.ones(9, np.float32)
    scale = np.array([0.05, 0.04, 0.03], np.float32)
    m.set_norm(mean, std, scale)
    xd, td = torch.from_numpy(X).cuda(), torch.from_numpy(T).cuda()
    gd = torch.empty(m.nparams, dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    loss = m.grad_dev(n, xd.data_ptr(), td.data_ptr(), gd.data_ptr())
    lo, go = M.loss_grad(p, mean, std, scale, X, T)
    rel = np.linalg.norm(gd.cpu().numpy() - go) / np.linalg.norm(go)
    print(f"{n} rows: gradient {rel:.2e}, loss {loss:.6e} vs {lo:.6e}", flush=True)
    # an FP32 sum on the other side of a BF16 rounding moves one activation by 2^-8 of
    # itself; few rows average few of them
    tol = 4e-3 if n < 64 else 1e-3
    assert rel < tol and abs(loss - lo) <= tol * lo


def test_gelu_range():
    """Inputs whose hidden pre-activations reach hundreds: finite, and the oracle's values."""
    import torch
    import rbc3d_amd as R
    m, p = _net(R, 6)
    X, _ = _data(9, 333)
    X *= np.logspace(-3, 3, 333, dtype=np.float32)[:, None]
    one = np.ones(9, np.float32)
    m.set_norm(0 * one, one, one[:3])
    xd = torch.from_numpy(X).cuda()
    yd = torch.empty((333, 3), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    m.forward_dev(333, xd.data_ptr(), yd.data_ptr())
    y, yo = yd.cpu().numpy().astype(np.float64), M.predict(p, 0 * one, one, one[:3], X)
    assert np.isfinite(y).all()
    # per row, against the row's scale (BF16 roundings that fall the other way)
    assert (np.abs(y - yo).max(1) <= 1e-2 * np.maximum(np.abs(yo).max(1), 1e-2)).all()
