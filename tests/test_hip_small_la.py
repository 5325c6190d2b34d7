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


@pytest.mark.parametrize("d", [1, 2, 3, 4])
@pytest.mark.parametrize("D", [2, 3, 4, 5, 6, 7, 8])
def test_bond_decompose_shapes(hip, D, d):
    """The register QR at every column count and wave layout (D^3 x d D, up to
    512 x 32, where the memory kernel takes over), each bond direction, against
    LAPACK.  m n half-ulps of the norm for the residual and for the
    orthonormality; R times the condition of its matrix more."""
    from oracle import full_update as ofu
    g = np.random.default_rng(10 * D + d)
    m, n = D ** 3, D * d
    for k in range(4):
        A1, A2 = (g.standard_normal((D, D, D, D, d)) for _ in range(2))
        a = [np.transpose(A, ofu.bond_permutation(k)) for A in (A1, A2)]
        ref = ofu.decompose_site_tensors(*a)
        out = [t.cpu().numpy() for t in hip.bond_decompose(
            torch.as_tensor(A1, device="cuda"), torch.as_tensor(A2, device="cuda"), k)]
        for i in (0, 2):
            assert out[i].shape == ref[i].shape
            q = out[i].reshape(m, n)
            assert np.abs(q.T @ q - np.eye(n)).max() <= m * n * 2.0 ** -53
            R = ref[i + 1]
            norm, cond = np.linalg.norm(R), np.linalg.cond(np.moveaxis(R, 1, 2).reshape(n, n))
            tol = m * n * 2.0 ** -53 * cond
            assert np.abs(out[i + 1] - R).max() <= tol * norm
            assert np.abs(out[i] - ref[i]).max() <= tol


@pytest.mark.parametrize("nD", [1, 2, 3, 4, 5, 6, 7, 8, 12, 16])
def test_gauge_fix_shapes(hip, nD):
    """The tall QR pair (nD^3 x nD, 1 to 4096 rows) behind the reduced gauge,
    through the pseudo-inverses of its factors, whose row signs are free.  The
    columns are Gaussian, so the condition stays below 100 for nD >= 2."""
    g = np.random.default_rng(nD)
    nz = g.standard_normal((nD, nD, nD * nD))
    a12g = g.standard_normal((nD, nD, 2, 2))
    _, _, xi, yi = [t.cpu().numpy() for t in hip.gauge_fix(
        torch.as_tensor(nz, device="cuda"), torch.as_tensor(a12g, device="cuda"), 1e-12)]
    for h, axis in ((xi, 1), (yi, 0)):
        A = np.moveaxis(nz, axis, -1).reshape(-1, nD)
        # pinv(R) pinv(R)^T = (A^T A)^-1
        exact = np.linalg.inv(A.T @ A)
        tol = 100 * nD ** 4 * 2.0 ** -53 * np.linalg.cond(A) ** 2
        assert np.abs(h @ h.T - exact).max() <= tol * np.abs(exact).max()


@pytest.mark.parametrize("case", ["full", "graded", "deficient", "equal"])
@pytest.mark.parametrize("n,scale", [(1, 1.0), (2, 1.0), (3, 1.0), (8, 1.0), (15, 1.0), (24, 1.0),
                                     (31, 1.0), (32, 1.0), (24, 1e-70), (24, 1e70)])
def test_small_svd_spectra(hip, n, scale, case):
    """The one-wave-a-pair Jacobi SVD of the bond update through the plain
    start, which returns U s^1/2 and V s^1/2 in units of s_0: products of both
    against the matrix, n^2 rotations' worth of rounding (60 n eps)."""
    s = {"full": np.linspace(1.0, 0.1, n), "graded": np.exp(-30.0 * np.arange(n) / n),
         "deficient": np.where(np.arange(n) < (n + 1) // 2, 1.0, 0.0) * np.linspace(1.0, 0.5, n),
         "equal": np.ones(n)}[case]
    g = np.random.default_rng(n)
    U = np.linalg.qr(g.standard_normal((n, n)))[0]
    V = np.linalg.qr(g.standard_normal((n, n)))[0]
    M = (U * s) @ V.T
    a12g = torch.as_tensor(M.reshape(n, n, 1, 1) * scale, device="cuda")
    a1, a2 = [t.cpu().numpy().reshape(n, n) for t in hip.als_initialize(a12g, n)]
    tol = 60 * n * 2.2e-16
    assert np.abs(a1 @ a2.T - M / s[0]).max() <= tol
    for a, W in ((a1, U), (a2, V)):
        assert np.abs(a.T @ a - np.diag(s / s[0])).max() <= tol


@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("K", [1, 15, 16, 17, 63, 64, 65, 315, 1023, 1025, 3071, 3072, 3073])
def test_small_gemm_tile_edges(hip, K, ta, tb):
    """The one-tile-a-workgroup FP64 product at the remainders of its tiles and
    k blocks, every operand order, one to sixteen waves and the first K past
    its range, against numpy: 2 eps K at most in units of the norms."""
    g = np.random.default_rng(K)
    for M, N in ((1, 1), (15, 17), (16, 16), (33, 66), (315, 37), (64, 129), (700, 5)):
        A = g.standard_normal((K, M) if ta else (M, K))
        B = g.standard_normal((N, K) if tb else (K, N))
        C = hip.gemm(torch.as_tensor(A, device="cuda"), torch.as_tensor(B, device="cuda"),
                     ta=ta, tb=tb).cpu().numpy()
        a, b = (A.T if ta else A), (B.T if tb else B)
        scale = np.linalg.norm(a, axis=1)[:, None] * np.linalg.norm(b, axis=0)
        assert np.all(np.abs(C - a @ b) <= 4.4e-16 * (K + 1) * scale), (M, N, K)


@pytest.mark.parametrize("sign", [1.0, -1.0])
@pytest.mark.parametrize("nD,D,d", [(1, 1, 1), (2, 1, 2), (3, 2, 1), (4, 2, 2), (5, 3, 3), (8, 4, 2),
                                    (9, 5, 1), (12, 4, 2), (7, 7, 1), (12, 6, 2), (10, 8, 1),
                                    (9, 9, 2), (16, 7, 2), (22, 5, 1), (15, 8, 1)])
def test_als_sweep_shapes(hip, nD, D, d, sign):
    """One ALS sweep at the edges of its tiles and of the register factor's
    three sizes (nD D up to 120), alone and in a batch, against numpy's solve.
    The norm is Gaussian with four samples a row, so the systems' condition
    stays near 10; a negative one takes the pivoted elimination.  2 nR^2
    half-ulps times the condition of each system, both in turn."""
    g = np.random.default_rng(100 * nD + 10 * D + d)
    n2, nR = nD * nD, nD * D
    M = g.standard_normal((n2, 4 * n2))
    N = (M @ M.T / (4 * n2) * sign).reshape(nD, nD, nD, nD)
    a12g = g.standard_normal((nD, nD, d, d))
    a1, a2 = g.standard_normal((nD, D, d)), g.standard_normal((nD, D, d))
    n12g = np.tensordot(N, a12g, ((0, 1), (0, 1)))                       # [Y, X, p, q]
    tol = 0.0
    for side in (0, 1):
        n, x, G = (N, a2, n12g) if side == 0 else (
            N.transpose(1, 0, 3, 2), a1, n12g.transpose(1, 0, 3, 2))
        t = np.tensordot(n, x, ((1,), (0,)))                             # [a, A, B, u, Q]
        R = np.tensordot(t, x, ((2, 4), (0, 2)))                         # [a, A, u, U]
        R = R.transpose(1, 3, 0, 2).reshape(nR, nR)
        S = np.tensordot(G, x, ((1, 3), (0, 2))).transpose(0, 2, 1).reshape(nR, d)
        R = 0.5 * (R + R.T)
        R = R + 1e-12 * np.abs(R).max() * np.eye(nR)
        X = np.linalg.solve(R, S).reshape(nD, D, d)
        tol += 2 * nR ** 2 * 2.0 ** -53 * np.linalg.cond(R)
        if side == 0:
            a1n, a1 = X, X
        else:
            a2n = X
    dv = lambda t: torch.as_tensor(t, device="cuda")
    start = g.standard_normal((nD, D, d))  # the first tensor's start does not enter
    h1, h2, _, _, flags = hip.als_solve(dv(N), dv(a12g), dv(start), dv(a2), 1, 1e-15, "cholesky",
                                        1e-12)
    assert flags == (0 if sign > 0 else 1)
    assert np.abs(h1.cpu().numpy() - a1n).max() <= tol * np.abs(a1n).max()
    assert np.abs(h2.cpu().numpy() - a2n).max() <= tol * np.abs(a2n).max()
    b1, b2, _, _, bf = hip.als_solve_batch(dv(N)[None].repeat(2, 1, 1, 1, 1),
                                           dv(a12g)[None].repeat(2, 1, 1, 1, 1), D, 1, 1e-15,
                                           "cholesky", 1e-12,
                                           (dv(start)[None].repeat(2, 1, 1, 1),
                                            dv(a2)[None].repeat(2, 1, 1, 1)))
    for i in (0, 1):
        assert torch.equal(b1[i], h1) and torch.equal(b2[i], h2) and int(bf[i]) == flags


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("d", [1, 2, 3])
@pytest.mark.parametrize("D", [1, 2, 3, 4, 5, 6, 7, 8])
def test_double_layer_shapes(hip, D, d, precision):
    """The double-layer absorption at every tile count and padding, fewer and
    more boundary blocks than waves, against the oracle's enlarged corner:
    one ulp (of FP32 in mixed precision, with the split corner's rounding) per
    term of the longest sum, in units of the sums of magnitudes."""
    from oracle import ctmrg as oc

    def raw(s):  # oracle.make_quarter_tensor before it is scaled
        a = oc.bond_permute(s["A"], 1)
        q = oc.ein("acuU,ealL->cuUelL", oc.ein("ab,bcuU->acuU", s["C"][1], s["E"][1]), s["E"][0])
        q = oc.ein("lurdp,cuelRDp->crRedD", a, oc.ein("cuUelL,LURDp->cuelRDp", q, a))
        return q.reshape(q.shape[0] * D * D, -1)

    rng = np.random.default_rng(10 * D + d)
    for chi in (3, 33) if D <= 4 else (3, 7):
        site = {"A": rng.standard_normal((D, D, D, D, d)),
                "C": [rng.standard_normal((chi, chi)) for _ in range(4)],
                "E": [rng.standard_normal((chi, chi, D, D)) for _ in range(4)]}
        mag = {k: np.abs(v) if k == "A" else [np.abs(t) for t in v] for k, v in site.items()}
        dv = lambda t: torch.as_tensor(t, device="cuda")
        try:
            got = hip.quarter_tensor((dv(site["A"]), [dv(t) for t in site["C"]],
                                      [dv(t) for t in site["E"]]), 1, precision=precision)
        except RuntimeError as e:
            assert "LDS budget" in str(e) and (D, d) == (8, 3) and precision == "fp64"
            continue
        got, ref, mg = got.cpu().numpy(), raw(site), raw(mag)
        sc = np.abs(ref).max() / np.abs(got).max()  # the engine's may be scaled
        ulp = 2.0 ** -52 if precision == "fp64" else 2.0 ** -23
        terms = 2 * chi + D ** 4 * d
        assert np.all(np.abs(got * sc - ref) <= 2 * ulp * terms * mg)


@pytest.mark.parametrize("rank", ["full", "half"])
@pytest.mark.parametrize("m,q", [(1, 1), (16, 1), (17, 16), (33, 17), (80, 22), (97, 32), (84, 33),
                                 (48, 45), (64, 39), (65, 40), (24, 64)])
def test_orthonormalize_small_bases(hip, m, q, rank):
    """The one-launch CholeskyQR at the remainders of its tiles and on both
    sides of its line (1e5 multiply-adds), with full and deficient columns,
    against LAPACK's spans (columns of condition 1e3: 1e-12)."""
    g = np.random.default_rng(m + q)
    q = min(m, q)
    r = q if rank == "full" else (q + 1) // 2
    Y = g.standard_normal((m, r)) * np.logspace(0, -3, r)
    Y = np.concatenate([Y, Y[:, :q - r] + Y[:, r - 1:r]], axis=1)
    Q = hip.orthonormalize(torch.as_tensor(Y, device="cuda")).cpu().numpy()
    assert np.abs(Q.T @ Q - np.eye(q)).max() <= 1e-13
    ref = np.linalg.qr(Y[:, :r])[0]
    for n in sorted({1, (r + 1) // 2, r}):
        P = ref[:, :n] - Q[:, :r] @ (Q[:, :r].T @ ref[:, :n])
        if rank == "half":
            P = ref[:, :n] - Q @ (Q.T @ ref[:, :n])
        assert np.abs(P).max() <= 1e-12


@pytest.mark.parametrize("chi,cd", [(1, 1), (2, 7), (16, 16), (17, 15), (64, 65), (64, 255),
                                    (127, 129), (128, 128), (128, 129), (181, 90), (256, 64)])
def test_renormalized_norms(hip, chi, cd):
    """The Frobenius normalisation at the edges of its blocks of 256 and on both
    sides of its one-launch range (64 of them), through the renormalised
    corners (chi x cd) and edge: unit norms to the rounding of a tree of sums
    and of one scaling, 20 ulps."""
    g = np.random.default_rng(chi + cd)
    dv = lambda *s: torch.as_tensor(g.standard_normal(s), device="cuda")
    D = 2
    site = (dv(D, D, D, D, 2), [dv(chi, chi) for _ in range(4)],
            [dv(chi, chi, D, D) for _ in range(4)])
    P = [dv(chi * D * D, cd) for _ in range(4)]
    out = hip.renormalize_boundary(site, 0, *P)
    for t in out:
        assert abs(float(torch.linalg.vector_norm(t.cpu())) - 1.0) <= 20 * 2.0 ** -52


@pytest.mark.parametrize("D,chi,projectors,bound", [(2, 4, "half-system", 4), (3, 16, "half-system", 0),
                                                    (2, 10, "full-system", 0)])
def test_default_start_is_not_computed_twice(hip, monkeypatch, D, chi, projectors, bound):
    """From the default start (a boundary of D^2, graded spectra) no pair is
    begun without the recovery of dropped columns and started over, over
    several calls of renormalize(); where the boundary is at chi from the
    first move on, the four pairs begun before anything is known are."""
    from acetn.ipeps import Ipeps
    made = []
    job = hip.ProjectorJob

    class Job(job):
        def __init__(self, *a, **kw):
            super().__init__(*a, **kw)
            made.append(self)
    monkeypatch.setattr(hip, "ProjectorJob", Job)
    torch.manual_seed(11)
    net = Ipeps({"TN": {"nx": 2, "ny": 2, "dims": {"phys": 2, "bond": D, "chi": chi}},
                 "ctmrg": {"steps": 1, "projectors": projectors, "sketch_seed": 3,
                           "disable_progressbar": True}})
    for _ in range(3):
        net.renormalize()
    assert len(made) == 3 * 16
    over = [i for i, j in enumerate(made) if j.started_over]
    assert len(over) <= bound and all(i < 4 for i in over)


@pytest.mark.parametrize("ta", [False, True])
@pytest.mark.parametrize("M,N,K", [(1040, 146, 1100), (5184, 146, 1234), (96, 50, 32838),
                                   (320, 48, 410)])
def test_gemm_keeps_infinities_where_they_belong(hip, M, N, K, ta):
    """An infinity in the last row of B (the one next to the padding of the last
    k-tile) makes its column infinite with the signs of A's last column, not
    undefined, and reaches no other; likewise one in A."""
    g = np.random.default_rng(K)
    A, B = g.standard_normal((M, K)), g.standard_normal((K, N))
    dv = lambda t: torch.as_tensor(np.ascontiguousarray(t), device="cuda")
    run = lambda a, b: hip.gemm(dv(a.T if ta else a), dv(b), ta=ta).cpu().numpy()
    Bi, Ai = B.copy(), A.copy()
    Bi[K - 1, N - 1] = np.inf
    C = run(A, Bi)
    assert np.array_equal(C[:, N - 1], np.sign(A[:, K - 1]) * np.inf)
    assert np.isfinite(C[:, :N - 1]).all()
    Ai[M - 1, K - 1] = -np.inf
    C = run(Ai, B)
    assert np.array_equal(C[M - 1], np.sign(B[K - 1]) * -np.inf)
    assert np.isfinite(C[:M - 1]).all()


@pytest.mark.parametrize("case", ["separate", "triples", "clusters", "graded"])
@pytest.mark.parametrize("q", [47, 48, 64, 97, 128, 129, 161, 192, 385, 448, 449, 464, 465])
def test_gram_svd_dispatch_lines(hip, q, case):
    """The same at the lines of the tridiagonal route (48 to 464), of its
    register kernel (192) and of its kernels by 32 and by 64 columns, those of
    the largest sizes among them."""
    test_gram_svd_spectra(hip, q, case)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("D", [1, 2, 3, 4, 5, 6, 7, 8])
def test_double_layer_absolute_values(hip, D, precision):
    """The enlarged corner itself, no scale fitted: the engine applies none.  The
    same bound as test_double_layer_shapes, through the oracle's corner times
    the largest element that it divides by."""
    from oracle import ctmrg as oc
    rng = np.random.default_rng(D)
    chi = 5
    site = {"A": rng.standard_normal((D, D, D, D, 2)),
            "C": [rng.standard_normal((chi, chi)) for _ in range(4)],
            "E": [rng.standard_normal((chi, chi, D, D)) for _ in range(4)]}

    def corner(s):
        a = oc.bond_permute(s["A"], 1)
        q = oc.ein("acuU,ealL->cuUelL", oc.ein("ab,bcuU->acuU", s["C"][1], s["E"][1]), s["E"][0])
        q = oc.ein("lurdp,cuelRDp->crRedD", a, oc.ein("cuUelL,LURDp->cuelRDp", q, a))
        return q.reshape(chi * D * D, -1)
    dv = lambda t: torch.as_tensor(t, device="cuda")
    got = hip.quarter_tensor((dv(site["A"]), [dv(t) for t in site["C"]],
                              [dv(t) for t in site["E"]]), 1, precision=precision).cpu().numpy()
    ref = corner(site)
    mag = corner({k: np.abs(v) if k == "A" else [np.abs(t) for t in v] for k, v in site.items()})
    ulp = 2.0 ** -52 if precision == "fp64" else 2.0 ** -23
    assert np.all(np.abs(got - ref) <= 2 * ulp * (2 * chi + 2 * D ** 4) * mag)
