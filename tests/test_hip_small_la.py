"""The one-workgroup factorisations at the edges of their tiles."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from acetn import _hip
    _hip.require_gpu()
    return _hip


@pytest.mark.parametrize("q", [1, 2, 15, 16, 17, 32, 33, 48, 49, 64, 65, 112, 113, 128, 129, 176,
                               177, 256, 257, 272, 273])
def test_orthonormalize_tile_edges(hip, q):
    """CholeskyQR at every change of tile count and wave layout, against the
    spans of LAPACK's Householder QR (columns of condition 1e3: the projector
    onto each leading block of columns agrees to 1e-12)."""
    g = np.random.default_rng(q)
    m = 2 * q + 37
    Y = g.standard_normal((m, q)) * np.logspace(0, -3, q)
    Q = hip.orthonormalize(torch.as_tensor(Y, device="cuda")).cpu().numpy()
    assert np.abs(Q.T @ Q - np.eye(q)).max() <= 1e-13
    ref = np.linalg.qr(Y)[0]
    for n in sorted({1, (q + 1) // 2, q}):
        P = Q[:, :n] - ref[:, :n] @ (ref[:, :n].T @ Q[:, :n])
        assert np.abs(P).max() <= 1e-12
