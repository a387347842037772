"""The association where it is decided in the last bits: candidates whose
squared distances differ by a few ulp around each other and around max_dist
(their rounded roots may be equal, and then the first one stays), and the
extreme values of max_dist; bit for bit against the oracle."""
import numpy as np
import pytest
import torch

from oracle import icp as oicp
from superscanner_amd import icp

pytestmark = pytest.mark.gpu

H, W, INTR = 45, 67, (60.0, 60.0, 33.0, 22.0)


def maps(seed):
    """x on the pixel rays at depth 1; y(k, l) at a distance from x's pixel that is one radius, give or take ulps."""
    rng = np.random.default_rng(seed)
    i, j = np.meshgrid(np.arange(H, dtype=np.float32), np.arange(W, dtype=np.float32), indexing="ij")
    x = np.stack([(j - 33.0) / 60.0, (i - (H - 22.0)) / 60.0, np.ones_like(i)], -1).astype(np.float32)
    y = np.repeat(x[22, 33][None], H * W, 0).reshape(H, W, 3).copy()  # all candidates around one point
    d = rng.normal(size=(H, W, 3))
    y += (0.05 * d / np.linalg.norm(d, axis=-1, keepdims=True)).astype(np.float32)
    y = (y.view(np.int32) + rng.integers(-2, 3, size=y.shape, dtype=np.int32)).view(np.float32)
    y[rng.random((H, W)) < 0.05] = 0.0
    n = rng.normal(size=(H, W, 3)).astype(np.float32)
    n /= np.linalg.norm(n, axis=-1, keepdims=True)
    n[rng.random((H, W)) < 0.05] = 0.0
    x[:] = x[22, 33]  # every pixel projects to the centre: one window for all
    x += (rng.integers(-8, 9, size=x.shape) * 2.0 ** -23).astype(np.float32)
    return x, y, n


@pytest.mark.parametrize("ns", [0, 1, 5, 8, 17])
@pytest.mark.parametrize("plane", [False, True])
def test_candidates_a_few_ulp_apart(gpu, ns, plane):
    x, y, n = maps(ns)
    dx, dy, dn = (torch.from_numpy(a).cuda() for a in (x, y, n))
    f = np.float32
    for md in (0.075, 0.05, float(np.nextafter(f(0.05), f(1))), float(np.nextafter(f(0.05), f(0))), 0.0, -0.075, 1e-12,
               1e-9, 1e-30, 2e6, float("inf"), float("nan")):
        got = icp.associate(dx, dy, dn, np.eye(4), INTR, int(plane), ns, md).cpu().numpy()
        exp = oicp.associate(x, y, n, np.eye(4), INTR, int(plane), ns, md)
        assert (got.view(np.int32) == exp.view(np.int32)).all(), (md, int((got != exp).any(-1).sum()))


def test_many_iterations_and_an_early_end(gpu):
    """More iterations than are queued at once, and iterations that end at the first without a correspondence."""
    rng = np.random.default_rng(3)
    d1 = torch.from_numpy(rng.integers(900, 1100, size=(H, W)).astype(np.int16)).cuda()
    T, rmse, fit = icp.kokkosICP(d1, d1, np.eye(4), np.eye(4), INTR, n_it=150)
    To, rmse_o, fit_o, _ = oicp.kokkosICP(d1.cpu().numpy().view(np.uint16), d1.cpu().numpy().view(np.uint16), np.eye(4),
                                          np.eye(4), INTR, n_it=150)
    assert np.abs(T - To).max() < 1e-5 and abs(rmse - rmse_o) <= 1e-5 * max(rmse_o, 1.0) and abs(fit - fit_o) < 1e-6
    far = np.eye(4)
    far[2, 3] = 50.0
    T, rmse, fit = icp.kokkosICP(d1, d1, far, np.eye(4), INTR, n_it=150)
    assert np.array_equal(T, np.eye(4)) and rmse == 1e6 and fit == 0.0
