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


@pytest.mark.parametrize("case", ["separate", "pairs", "triples", "clusters", "equal", "graded",
                                  "deficient"])
@pytest.mark.parametrize("q", [1, 2, 9, 31, 32, 33, 65, 96, 130, 160, 193, 300])
def test_gram_svd_spectra(hip, q, case):
    """The Gram-matrix SVD behind the projectors at the edges of the
    tridiagonal kernels' blocks, on spectra of every kind.  A Jacobi solve
    takes each column through q - 1 rotations a sweep, each good to 3 eps, and
    some twelve sweeps in its two passes: 36 eps q = 4e-15 q for the
    orthonormality of the vectors, the same for the values in units of s_0
    (sqrt(eps) where they vanish).  The projector onto each group of equal
    values is compared where the values are resolved: eps s_0 / (s gap), with
    gaps of 0.02 and more, times the q terms of its entries."""
    i = np.arange(q)
    s = np.exp(-7.0 * i / max(q, 2))
    if case in ("pairs", "triples"):
        n = 2 if case == "pairs" else 3
        s = s[i // n * n]
    elif case == "clusters":
        s = s[i // 7 * 7] * (1.0 - 1e-9 * (i % 7))
    elif case == "equal":
        s = np.ones(q)
    elif case == "graded":
        s = np.exp(-23.0 * i / max(q, 2))
    elif case == "deficient":
        s = np.where(i < (q + 1) // 2, s, 0.0)
    g = np.random.default_rng(100 * q + len(case))
    U = np.linalg.qr(g.standard_normal((q, q)))[0]
    V = np.linalg.qr(g.standard_normal((700, q)))[0]
    w, UB = hip.gram_svd(torch.as_tensor(V @ (U * s).T, device="cuda"))
    sv, UB = torch.sqrt(torch.clamp(w, min=0.0)).cpu().numpy(), UB.cpu().numpy()
    tol = 4e-15 * q + 1e-15
    assert np.abs(sv - s).max() <= (1.5e-8 * q if case == "deficient" else tol)
    assert np.abs(UB.T @ UB - np.eye(q)).max() <= tol
    new = np.concatenate([[True], s[1:] < s[:-1] * (1.0 - 1e-6)])
    group = np.cumsum(new) - 1
    for k in range(group[-1] + 1):
        at = np.nonzero(group == k)[0]
        if s[at[0]] < 1e-6:
            continue
        P, R = UB[:, at] @ UB[:, at].T, U[:, at] @ U[:, at].T
        assert np.abs(P - R).max() <= 2.2e-16 * q / (0.02 * s[at[0]])


@pytest.mark.parametrize("start", ["product", "random"])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_trusted_range_finder_starts_over(hip, start, precision):
    """A pair begun without the launches that deal with dropped columns ends
    with the bits of one begun with them: on a graded spectrum (columns are
    dropped: the count comes back -1 and the pair starts over) and on one that
    drops none (a count at once)."""
    from oracle import ctmrg as oc
    from test_hip_ctmrg import product_start, to_dev_site
    D, chi = (4, 16) if start == "product" else (3, 9)
    st = product_start(D, 5) if start == "product" else \
        oc.make_state(oc.random_site_tensors(2, 2, D, 2, seed=41))
    dsites = [to_dev_site(st[s]) for s in oc.plaquette(2, 2, 0, 1, 0)]
    out, counts = [], []
    for trust in (False, True):
        job = hip.ProjectorJob(0, dsites, 0, chi, 2, 2, 1e-12, 21, 3, precision=precision,
                               trust=trust)
        job.ready.synchronize()
        counts.append(int(job.cd_host[0]))
        P1, P2 = job.finish()
        torch.cuda.synchronize()
        out.append((P1.cpu(), P2.cpu(), job.spec.cpu(), job.spec_host.clone()))
    assert counts[0] > 0
    assert counts[1] == (-1 if start == "product" else counts[0])
    for a, b in zip(*out):
        assert torch.equal(a, b)


@pytest.mark.parametrize("ta", [False, True])
@pytest.mark.parametrize("N", [17, 18, 33, 50, 66, 82, 98, 114, 130, 146, 160, 162, 258, 322])
def test_large_gemm_tile_edges(hip, N, ta):
    """The pipelined FP64 product at every tile width, with remainders of rows,
    columns and k (odd sizes among them) and one or several k parts, against
    numpy: K terms of unit variance, 2 eps K at most in units of their
    norms."""
    g = np.random.default_rng(N)
    for M, K in ((96, 32768 + 2 * N), (1030, 3000), (1031, 3001), (4098, 1234), (9000, 402)):
        A = g.standard_normal((K, M) if ta else (M, K))
        B = g.standard_normal((K, N))
        C = hip.gemm(torch.as_tensor(A, device="cuda"), torch.as_tensor(B, device="cuda"),
                     ta=ta).cpu().numpy()
        exact = (A.T if ta else A) @ B
        scale = np.linalg.norm(A, axis=0 if ta else 1)[:, None] * np.linalg.norm(B, axis=0)
        assert np.all(np.abs(C - exact) <= 4.4e-16 * K * scale), (M, N, K)
