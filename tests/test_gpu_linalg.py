"""Dense complex128 kernels (ZGEMM, LU, solve, eigensolver) against numpy/LAPACK."""
import ctypes as C

import numpy as np
import pytest

from varrcwa_amd._lib import cplx, from_dev_colmajor, ptr, to_dev_colmajor

pytestmark = pytest.mark.gpu


def crand(rng, *shape):
    return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)


def opm(a, op):
    return a if op == 0 else (np.swapaxes(a, -1, -2) if op == 1 else np.conj(np.swapaxes(a, -1, -2)))


@pytest.mark.parametrize("opA", [0, 1, 2])
@pytest.mark.parametrize("opB", [0, 1, 2])
def test_zgemm_ops(ctx, opA, opB):
    rng = np.random.default_rng(10 * opA + opB)
    m, n, k, batch = 70, 45, 37, 3
    A = crand(rng, batch, *((m, k) if opA == 0 else (k, m)))
    B = crand(rng, batch, *((k, n) if opB == 0 else (n, k)))
    Cm = crand(rng, batch, m, n)
    alpha, beta = 0.7 - 0.2j, -0.3 + 1.1j
    dA, dB, dC = to_dev_colmajor(A), to_dev_colmajor(B), to_dev_colmajor(Cm)
    lda, ldb = A.shape[1], B.shape[1]
    ctx.check(ctx.lib.vrc_zgemm(ctx.h, opA, opB, m, n, k, cplx(alpha), ptr(dA), lda, A.shape[1] * A.shape[2],
                                ptr(dB), ldb, B.shape[1] * B.shape[2], cplx(beta), ptr(dC), m, m * n, batch),
              "zgemm")
    ref = alpha * (opm(A, opA) @ opm(B, opB)) + beta * Cm
    got = from_dev_colmajor(dC)
    assert np.abs(got - ref).max() <= 1e-13 * np.abs(ref).max()


@pytest.mark.parametrize("opA,opB", [(0, 0), (2, 0), (0, 2), (1, 1)])
@pytest.mark.parametrize("m,n,k,batch", [(1, 1, 1, 1), (16, 17, 15, 2), (31, 33, 32, 3), (33, 64, 65, 1),
                                         (97, 49, 31, 40), (65, 81, 16, 130), (98, 98, 33, 300)])
def test_zgemm_tile_edges(ctx, opA, opB, m, n, k, batch):
    """Both ZGEMM tiles at the edges of their 16x16 blocks, of their K chunks (16, 32) and of
    the rule that picks one (few workgroups: 32x32, many: 64x64), NaN in C with beta = 0."""
    import torch
    rng = np.random.default_rng(m + 100 * n + k)
    A = crand(rng, batch, *((m, k) if opA == 0 else (k, m)))
    B = crand(rng, batch, *((k, n) if opB == 0 else (n, k)))
    dA, dB = to_dev_colmajor(A), to_dev_colmajor(B)
    dC = torch.full((batch, n, m), float("nan"), dtype=torch.complex128, device="cuda")
    ctx.check(ctx.lib.vrc_zgemm(ctx.h, opA, opB, m, n, k, cplx(1), ptr(dA), A.shape[1], A.shape[1] * A.shape[2],
                                ptr(dB), B.shape[1], B.shape[1] * B.shape[2], cplx(0), ptr(dC), m, m * n, batch),
              "zgemm")
    ref = opm(A, opA) @ opm(B, opB)
    assert np.abs(from_dev_colmajor(dC) - ref).max() <= 1e-13 * np.abs(ref).max()


def test_zgemm_large_and_beta0(ctx):
    rng = np.random.default_rng(1)
    m = n = k = 300
    A, B = crand(rng, 2, m, k), crand(rng, 2, k, n)
    dA, dB = to_dev_colmajor(A), to_dev_colmajor(B)
    import torch
    dC = torch.full((2, n, m), float("nan"), dtype=torch.complex128, device="cuda")
    ctx.check(ctx.lib.vrc_zgemm(ctx.h, 0, 0, m, n, k, cplx(1), ptr(dA), m, m * k, ptr(dB), k, k * n, cplx(0),
                                ptr(dC), m, m * n, 2), "zgemm")
    ref = A @ B
    assert np.abs(from_dev_colmajor(dC) - ref).max() <= 1e-13 * np.abs(ref).max()


@pytest.mark.parametrize("n", [5, 33, 64, 130, 242])
def test_getrf_getrs(ctx, n):
    import torch
    rng = np.random.default_rng(n)
    batch, nrhs = 3, 2 * n + 3
    A = crand(rng, batch, n, n)
    B = crand(rng, batch, n, nrhs)
    dA, dB = to_dev_colmajor(A), to_dev_colmajor(B)
    ipiv = torch.zeros((batch, n), dtype=torch.int32, device="cuda")
    info = torch.zeros(batch, dtype=torch.int32, device="cuda")
    ctx.check(ctx.lib.vrc_zgetrf(ctx.h, n, ptr(dA), n, n * n, ptr(ipiv), n, ptr(info), batch), "getrf")
    dX = torch.zeros_like(dB)
    ctx.check(ctx.lib.vrc_zgetrs(ctx.h, n, nrhs, ptr(dA), n, n * n, ptr(ipiv), n, ptr(dB), n, n * nrhs,
                                 ptr(dX), n, n * nrhs, batch), "getrs")
    X = from_dev_colmajor(dX)
    ref = np.linalg.solve(A, B)
    assert info.cpu().numpy().tolist() == [0] * batch
    err = np.abs(X - ref).max() / np.abs(ref).max()
    assert err < 1e-11, err
    # in-place solve (X aliases B)
    ctx.check(ctx.lib.vrc_zgetrs(ctx.h, n, nrhs, ptr(dA), n, n * n, ptr(ipiv), n, ptr(dB), n, n * nrhs,
                                 ptr(dB), n, n * nrhs, batch), "getrs in place")
    assert np.abs(from_dev_colmajor(dB) - ref).max() / np.abs(ref).max() < 1e-11


@pytest.mark.parametrize("n", [130, 1030])
def test_getrf_matches_lapack(ctx, n):
    """Pivot sequence and factors equal LAPACK zgetrf's (scipy lu_factor). n = 130 runs the
    register-resident panel (n <= 1024), n = 1030 the workgroup-per-panel kernel."""
    import torch
    from scipy.linalg import lu_factor
    rng = np.random.default_rng(7 + n)
    batch = 2
    A = crand(rng, batch, n, n)
    dA = to_dev_colmajor(A)
    ipiv = torch.zeros((batch, n), dtype=torch.int32, device="cuda")
    info = torch.zeros(batch, dtype=torch.int32, device="cuda")
    ctx.check(ctx.lib.vrc_zgetrf(ctx.h, n, ptr(dA), n, n * n, ptr(ipiv), n, ptr(info), batch), "getrf")
    LU = from_dev_colmajor(dA)
    piv = ipiv.cpu().numpy()
    assert info.cpu().numpy().tolist() == [0] * batch
    for b in range(batch):
        lu_ref, piv_ref = lu_factor(A[b])
        assert np.array_equal(piv[b], piv_ref), np.nonzero(piv[b] != piv_ref)[0][:5]
        assert np.abs(LU[b] - lu_ref).max() <= 1e-11 * np.abs(lu_ref).max()


@pytest.mark.parametrize("kind", ["dense", "ties"])
@pytest.mark.parametrize("n,batch", [(1, 2), (15, 3), (16, 2), (17, 5), (63, 2), (65, 2), (127, 1), (129, 3),
                                     (256, 1), (257, 2), (513, 1), (1024, 1)])
def test_getrf_panel_edges(ctx, n, batch, kind):
    """Backward error of the factors and of a solve at the edges of the panels (16), diagonal
    blocks (64), outer blocks (128) and panel thread counts (256, 512, 1024); "ties" has many
    equal pivot candidates. Bound: |P A - L U| <= gamma_n |L| |U|, gamma_n = 2 sqrt(2) n eps for
    complex products, here with 4 n eps; the solve's with the two triangular solves (three times
    that, and inverted 64-blocks whose condition the well-scaled factors keep below n)."""
    import torch
    rng = np.random.default_rng(n + batch)
    A = crand(rng, batch, n, n)
    if kind == "ties":
        A = np.round(A) + 0j
        A[:, np.arange(n), np.arange(n)] += 0.5
    dA = to_dev_colmajor(A)
    ipiv = torch.zeros(batch, n, dtype=torch.int32, device="cuda")
    info = torch.zeros(batch, dtype=torch.int32, device="cuda")
    ctx.check(ctx.lib.vrc_zgetrf(ctx.h, n, ptr(dA), n, n * n, ptr(ipiv), n, ptr(info), batch), "getrf")
    assert int(info.abs().max()) == 0
    LU, pv = from_dev_colmajor(dA), ipiv.cpu().numpy()
    eps = np.finfo(float).eps
    for b in range(batch):
        L, U = np.tril(LU[b], -1) + np.eye(n), np.triu(LU[b])
        PA = A[b].copy()
        for i, p in enumerate(pv[b]):
            assert i <= p < n
            PA[[i, p]] = PA[[p, i]]
        assert np.abs(np.tril(LU[b], -1)).max(initial=0.0) <= np.sqrt(2) * (1 + 1e-12)
        assert np.all(np.abs(PA - L @ U) <= 4 * n * eps * (np.abs(L) @ np.abs(U)))
    x = crand(rng, batch, n, 3)
    dB, dX = to_dev_colmajor(A @ x), to_dev_colmajor(x * 0)
    ctx.check(ctx.lib.vrc_zgetrs(ctx.h, n, 3, ptr(dA), n, n * n, ptr(ipiv), n, ptr(dB), n, 3 * n, ptr(dX), n, 3 * n,
                                 batch), "getrs")
    X = from_dev_colmajor(dX)
    for b in range(batch):
        r = np.abs(A[b] @ X[b] - A[b] @ x[b]).max()
        bound = np.abs(np.tril(LU[b], -1) + np.eye(n)) @ np.abs(np.triu(LU[b])) @ np.abs(X[b])
        assert r <= 12 * n * n * eps * bound.max()


@pytest.mark.parametrize("n", [1, 4, 31, 32, 33, 47, 48, 49, 80, 96, 97, 112, 113])
def test_getrs_last_block(ctx, n):
    """Solves whose last 64-row diagonal block holds one to four runs of 16 rows: the backward
    error of two triangular solves through inverted blocks, with the bound of the test above."""
    import torch
    rng = np.random.default_rng(900 + n)
    A, x = crand(rng, 2, n, n), crand(rng, 2, n, 5)
    dA = to_dev_colmajor(A)
    ipiv = torch.zeros(2, n, dtype=torch.int32, device="cuda")
    info = torch.zeros(2, dtype=torch.int32, device="cuda")
    ctx.check(ctx.lib.vrc_zgetrf(ctx.h, n, ptr(dA), n, n * n, ptr(ipiv), n, ptr(info), 2), "getrf")
    dB, dX = to_dev_colmajor(A @ x), to_dev_colmajor(x * 0)
    ctx.check(ctx.lib.vrc_zgetrs(ctx.h, n, 5, ptr(dA), n, n * n, ptr(ipiv), n, ptr(dB), n, 5 * n, ptr(dX), n, 5 * n, 2),
              "getrs")
    LU, X = from_dev_colmajor(dA), from_dev_colmajor(dX)
    eps = np.finfo(float).eps
    for b in range(2):
        r = np.abs(A[b] @ X[b] - A[b] @ x[b]).max()
        bound = np.abs(np.tril(LU[b], -1) + np.eye(n)) @ np.abs(np.triu(LU[b])) @ np.abs(X[b])
        assert r <= 12 * n * n * eps * bound.max()


def test_getrf_zero_column_info(ctx):
    """A zero column inside a panel: info names it (1-based), as LAPACK's."""
    import torch
    from scipy.linalg import lapack
    rng = np.random.default_rng(3)
    n = 70
    A = crand(rng, n, n)
    A[:, 37] = 0.0
    dA = to_dev_colmajor(A[None])
    ipiv = torch.zeros((1, n), dtype=torch.int32, device="cuda")
    info = torch.zeros(1, dtype=torch.int32, device="cuda")
    ctx.check(ctx.lib.vrc_zgetrf(ctx.h, n, ptr(dA), n, n * n, ptr(ipiv), n, ptr(info), 1), "getrf")
    _, _, info_ref = lapack.zgetrf(A)
    assert int(info.cpu()[0]) == info_ref == 38


def test_getrf_singular_info(ctx):
    import torch
    n = 6
    A = np.eye(n, dtype=complex)
    A[3, 3] = 0.0
    dA = to_dev_colmajor(A[None])
    ipiv = torch.zeros((1, n), dtype=torch.int32, device="cuda")
    info = torch.zeros(1, dtype=torch.int32, device="cuda")
    ctx.check(ctx.lib.vrc_zgetrf(ctx.h, n, ptr(dA), n, n * n, ptr(ipiv), n, ptr(info), 1), "getrf")
    assert int(info.cpu()[0]) == 4


def _eig_check(ctx, A, tol_res=1e-12):
    import torch
    batch, n, _ = A.shape
    dA = to_dev_colmajor(A)
    w = torch.zeros((batch, n), dtype=torch.complex128, device="cuda")
    VR = torch.zeros_like(dA)
    info = torch.zeros(batch, dtype=torch.int32, device="cuda")
    ctx.check(ctx.lib.vrc_zgeev(ctx.h, n, ptr(dA), n, n * n, ptr(w), n, ptr(VR), n, n * n, ptr(info), batch),
              "zgeev")
    ctx.sync()
    assert info.cpu().numpy().tolist() == [0] * batch
    W = w.cpu().numpy()
    V = from_dev_colmajor(VR)
    for b in range(batch):
        nrm = np.linalg.norm(A[b], 2)
        res = np.abs(A[b] @ V[b] - V[b] * W[b][None, :]).max() / nrm
        assert res < tol_res * n, (b, res)
        # unit norm, largest component real and positive
        assert np.allclose(np.linalg.norm(V[b], axis=0), 1.0, atol=1e-12)
        k = np.argmax(np.abs(V[b]) ** 2, axis=0)
        big = V[b][k, np.arange(n)]
        assert np.all(np.abs(big.imag) == 0) and np.all(big.real > 0)
        # eigenvalues vs LAPACK (sorted, well separated for random matrices)
        ref = np.linalg.eigvals(A[b])
        key = lambda z: np.lexsort((np.round(z.imag, 6), np.round(z.real, 6)))
        a, r = np.sort_complex(W[b]), np.sort_complex(ref)
        assert np.abs(a - r).max() / np.abs(r).max() < 1e-11
    return W, V


@pytest.mark.parametrize("n", [3, 20, 48, 49, 97, 200])
def test_zgeev_random(ctx, n):
    rng = np.random.default_rng(1000 + n)
    _eig_check(ctx, crand(rng, 2, n, n))


def test_zgeev_triangular_and_diag(ctx):
    rng = np.random.default_rng(5)
    n = 80
    A = np.triu(crand(rng, n, n))
    D = np.diag(crand(rng, n))
    _eig_check(ctx, np.stack([A, D]))


@pytest.mark.parametrize("variant", [1, 2, 4])
@pytest.mark.parametrize("n", [20, 49, 97, 200, 441])
def test_zgeev_qr_kernel_variants(ctx, variant, n):
    """The other QR kernel configurations of "zgeev.qr_variant": 1 (64-wide window, window
    products staged through LDS), 2 (48-wide window on 256 threads, two matrices per CU),
    4 (32-wide window on 128 threads, four per CU) against LAPACK eigenvalues and
    eigen-residuals, like the default kernel."""
    rng = np.random.default_rng(2000 + n)
    A = crand(rng, 3, n, n)
    assert ctx.lib.vrc_tune_set(b"zgeev.qr_variant", variant) == 0
    try:
        _eig_check(ctx, A)
    finally:
        assert ctx.lib.vrc_tune_set(b"zgeev.qr_variant", -1) == 0


@pytest.mark.parametrize("variant", [0, 2, 4])
@pytest.mark.parametrize("n", [2, 4, 31, 32, 33, 47, 50, 63, 64, 66])
def test_zgeev_window_edges(ctx, variant, n):
    """Sizes at the edges of the QR kernels' windows (32, 48, 64) and of the single-wavefront
    Schur form's two lane layouts (32), with entries of order one, entries whose squares leave
    the range of the fast rotations (1e140, 1e-140), and a cyclic shift (rotations with an
    exactly zero first entry)."""
    rng = np.random.default_rng(3000 + n)
    A = crand(rng, 2, n, n)
    shift = np.roll(np.eye(n), 1, axis=0).astype(complex)
    assert ctx.lib.vrc_tune_set(b"zgeev.qr_variant", variant) == 0
    try:
        for scale in (1.0, 1e140, 1e-140):
            _eig_check(ctx, A * scale)
        w, _ = _eig_check_values(ctx, shift[None])
        assert np.abs(w[0] ** n - 1.0).max() < 1e-12 * n * n
    finally:
        assert ctx.lib.vrc_tune_set(b"zgeev.qr_variant", -1) == 0


@pytest.mark.parametrize("n", [5, 50, 98])
def test_zgeev_defective(ctx, n):
    """Nilpotent Jordan blocks: one eigenvector for n equal eigenvalues, so the back substitution of
    the others overflows. The eigenvalues of these triangular matrices are their diagonal, every
    finite vector is an eigenvector, and a vector without a finite component is NaN throughout."""
    import torch
    for A in (np.diag(np.ones(n - 1), 1) + 0j, np.diag(np.ones(n - 1), 1) + 2.0 * np.eye(n)):
        dA = to_dev_colmajor(A[None])
        w = torch.zeros((1, n), dtype=torch.complex128, device="cuda")
        VR = torch.zeros_like(dA)
        info = torch.zeros(1, dtype=torch.int32, device="cuda")
        ctx.check(ctx.lib.vrc_zgeev(ctx.h, n, ptr(dA), n, n * n, ptr(w), n, ptr(VR), n, n * n, ptr(info), 1), "zgeev")
        ctx.sync()
        assert int(info[0]) == 0
        assert np.array_equal(np.sort_complex(w.cpu().numpy()[0]), np.sort_complex(np.diag(A)))
        V = from_dev_colmajor(VR)[0]
        ok = np.isfinite(V).all(axis=0)
        assert ok[0]
        assert np.abs(A @ V[:, ok] - V[:, ok] * w.cpu().numpy()[0][ok]).max() < 1e-12 * n
        assert np.isnan(V[:, ~ok]).all()


@pytest.mark.parametrize("n,batch", [(98, 513), (300, 2), (300, 60), (530, 65)])
@pytest.mark.parametrize("tiny", [1e-170, 1e-200])
def test_zgeev_tiny_coupling(ctx, n, batch, tiny):
    """Eigenvalues of order one coupled by entries whose squares underflow: the reflector of such a
    column has to be unitary all the same, in the Hessenberg panel of one workgroup per matrix
    (256, 512 and 1024 threads) and in the one spread over workgroups (300, 2)."""
    rng = np.random.default_rng(9000 + n)
    A = tiny * crand(rng, 1, n, n)
    A[:, np.arange(n), np.arange(n)] = np.arange(n)
    w, V = _eig_values(ctx, A, batch)
    for b in (0, batch - 1):
        assert np.abs(np.sort(w[b].real) - np.arange(n)).max() < 1e-13 * n
        assert np.abs(np.linalg.norm(V[b], axis=0) - 1.0).max() < 1e-13 * n
        assert np.abs(A[0] @ V[b] - V[b] * w[b][None, :]).max() < 1e-12 * n * n


def _eig_check_values(ctx, A):
    """Eigenvalues and vectors with the residual checked (no comparison of sorted spectra:
    eigenvalues of one modulus sort arbitrarily)."""
    import torch
    batch, n, _ = A.shape
    dA = to_dev_colmajor(A)
    w = torch.zeros((batch, n), dtype=torch.complex128, device="cuda")
    VR = torch.zeros_like(dA)
    info = torch.zeros(batch, dtype=torch.int32, device="cuda")
    ctx.check(ctx.lib.vrc_zgeev(ctx.h, n, ptr(dA), n, n * n, ptr(w), n, ptr(VR), n, n * n, ptr(info), batch),
              "zgeev")
    ctx.sync()
    assert info.cpu().numpy().tolist() == [0] * batch
    W, V = w.cpu().numpy(), from_dev_colmajor(VR)
    for b in range(batch):
        assert np.abs(A[b] @ V[b] - V[b] * W[b][None, :]).max() < 1e-12 * n * np.linalg.norm(A[b], 2)
    return W, V


@pytest.mark.parametrize("n", [200, 242])
def test_zgeev_team_sizes(ctx, n):
    """Launches of 1, 9, 40, 70 and 128 matrices give the QR kernel teams of 16, 16, 6, 3 and 2
    workgroups per matrix, 129 none: the same matrix gives the same bits whatever the team (the
    shares of a window product do not depend on who computes them)."""
    rng = np.random.default_rng(4000 + n)
    A = crand(rng, 1, n, n)
    ref = None
    for batch in (1, 9, 40, 64, 129, 70, 128):
        w, V = _eig_check_values(ctx, np.repeat(A, batch, axis=0)) if batch < 9 else _eig_values(ctx, A, batch)
        if ref is None:
            ref = (w[0], V[0])
        for b in (0, batch // 2, batch - 1):
            assert np.array_equal(w[b], ref[0]) and np.array_equal(V[b], ref[1]), (batch, b)


@pytest.mark.parametrize("n,batches", [(338, (1, 9, 40)), (338, (129, 64, 70, 128)), (450, (1, 9, 40, 64)),
                                       (450, (129, 70, 128))])
def test_zgeev_team_hand_over(ctx, n, batches):
    """Windows of many strips handed between the workgroups of a team, at sizes that are no
    multiple of the strips' 16: three different matrices in turn, each with the same bits in teams
    of 16, 16, 6 and 4 workgroups, and in teams of 4, 3 and 2 as in none (129 matrices). Few matrices
    and many take different forms of the Hessenberg panel, hence two groups."""
    import torch
    rng = np.random.default_rng(7000 + n)
    A = to_dev_colmajor(crand(rng, 3, n, n))
    ref = None
    for batch in batches:
        pick = torch.arange(batch, device="cuda") % 3
        dA = A[pick].contiguous()
        w = torch.zeros((batch, n), dtype=torch.complex128, device="cuda")
        VR = torch.zeros_like(dA)
        info = torch.zeros(batch, dtype=torch.int32, device="cuda")
        ctx.check(ctx.lib.vrc_zgeev(ctx.h, n, ptr(dA), n, n * n, ptr(w), n, ptr(VR), n, n * n, ptr(info), batch),
                  "zgeev")
        ctx.sync()
        assert int(info.abs().max()) == 0
        first = min(batch, 3)
        if ref is None or len(ref[0]) < first:
            assert ref is None or (torch.equal(w[:1], ref[0]) and torch.equal(VR[:1], ref[1]))
            ref = (w[:first].clone(), VR[:first].clone())
        assert torch.equal(w, ref[0][pick]) and torch.equal(VR, ref[1][pick]), batch
    B = from_dev_colmajor(A)
    V, W = from_dev_colmajor(ref[1]), ref[0].cpu().numpy()
    for b in range(len(V)):
        assert np.abs(B[b] @ V[b] - V[b] * W[b][None, :]).max() < 1e-12 * n * np.linalg.norm(B[b], 2)


def test_zgeev_team_streams(ctx):
    """Contexts on several streams divide the CUs between their teams (16 workgroups per matrix with
    one, 8, 5 and 4 with two to four): the bits stay the same, alone and with all contexts at
    work at once."""
    import threading

    import torch
    from varrcwa_amd._lib import Context
    rng = np.random.default_rng(4900)
    n, batch = 242, 8
    A = to_dev_colmajor(crand(rng, batch, n, n))
    out = {}

    def solve(key, c, stream):
        with torch.cuda.stream(stream):
            dA = A.clone()
            w = torch.zeros((batch, n), dtype=torch.complex128, device="cuda")
            VR = torch.zeros_like(dA)
            info = torch.zeros(batch, dtype=torch.int32, device="cuda")
            rc = c.lib.vrc_zgeev(c.h, n, ptr(dA), n, n * n, ptr(w), n, ptr(VR), n, n * n, ptr(info), batch)
            c.sync()
            out[key] = (rc, int(info.abs().max()), w.cpu().numpy(), VR.cpu().numpy())

    torch.cuda.synchronize()
    solve("one", ctx, torch.cuda.current_stream())
    streams = [torch.cuda.Stream() for _ in range(3)]
    more = []
    try:
        for s in streams:
            more.append(Context(0, s.cuda_stream))
            solve(len(more), ctx, torch.cuda.current_stream())
        threads = [threading.Thread(target=solve, args=(("thread", k), c, s)) for k, (c, s) in
                   enumerate(zip(more, streams))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    finally:
        for c in more:
            c.close()
    solve("after", ctx, torch.cuda.current_stream())
    assert len(out) == 8
    for key, (rc, bad, w, V) in out.items():
        assert rc == 0 and bad == 0, key
        assert np.array_equal(w, out["one"][2]) and np.array_equal(V, out["one"][3]), key


@pytest.mark.parametrize("n", [3, 17, 66, 67, 130, 162])
def test_zgeev_wide_hessenberg(ctx, n):
    """Up to 512 matrices take the Hessenberg panel with more loads in flight, more of them the
    one with four workgroups per CU: the sums are the same, so are the bits. Sizes at the edges
    of its column groups (8, 16), rows (64) and panels (64)."""
    rng = np.random.default_rng(6000 + n)
    A = crand(rng, 1, n, n)
    assert ctx.lib.vrc_tune_set(b"zgeev.qr_variant", 4) == 0
    try:
        few, many = _eig_values(ctx, A, 2), _eig_values(ctx, A, 513)
    finally:
        ctx.lib.vrc_tune_set(b"zgeev.qr_variant", -1)
    for b in (0, 512):
        assert np.array_equal(few[0][0], many[0][b]) and np.array_equal(few[1][0], many[1][b])
    _eig_check(ctx, A)


@pytest.mark.parametrize("n", [200, 257, 258, 259, 322])
def test_zgeev_spread_hessenberg(ctx, n):
    """The Hessenberg panel spread over workgroups (from N = 258) at the edges of its row blocks,
    column tiles and panels (64), and the largest sizes that are not spread, with identity
    reflectors (triangular input) in the batch."""
    rng = np.random.default_rng(5000 + n)
    A = crand(rng, 3, n, n)
    A[1] = np.triu(A[1]) + 3.0 * np.diag(np.arange(n))
    A[2, n // 2:, : n // 2] = 0.0
    _eig_check_values(ctx, A)
    _eig_check(ctx, A[:1])


@pytest.mark.parametrize("n,batch", [(258, 23), (322, 46), (373, 64), (500, 64)])
def test_zgeev_spread_line(ctx, n, batch):
    """The last count of matrices whose Hessenberg panel is spread over workgroups, and one more, in
    one workgroup each: sums in another order, so the eigenvalues agree to the rounding of the
    reduction (backward error n eps |A|, condition numbers of a random matrix below 1e4) and the
    residuals stay as small; with the spread one some matrices differ in the last bits."""
    rng = np.random.default_rng(8000 + n)
    A = crand(rng, 1, n, n)
    (w0, V0), (w1, V1) = _eig_values(ctx, A, batch), _eig_values(ctx, A, batch + 1)
    size = np.linalg.norm(A[0], 2)
    for w, V in ((w0, V0), (w1, V1)):
        assert np.array_equal(w[0], w[-1]) and np.array_equal(V[0], V[-1])
        assert np.abs(A[0] @ V[0] - V[0] * w[0][None, :]).max() < 1e-12 * n * size
    d = np.abs(w0[0][:, None] - w1[0][None, :])
    assert len(set(d.argmin(axis=1))) == n
    assert d.min(axis=1).max() < 1e4 * n * np.finfo(float).eps * size
    assert not np.array_equal(w0[0], w1[0])  # the two forms, not one of them twice


def _eig_values(ctx, A, batch):
    import torch
    n = A.shape[-1]
    dA = to_dev_colmajor(A).expand(batch, n, n).contiguous()
    w = torch.zeros((batch, n), dtype=torch.complex128, device="cuda")
    VR = torch.zeros_like(dA)
    info = torch.zeros(batch, dtype=torch.int32, device="cuda")
    ctx.check(ctx.lib.vrc_zgeev(ctx.h, n, ptr(dA), n, n * n, ptr(w), n, ptr(VR), n, n * n, ptr(info), batch),
              "zgeev")
    ctx.sync()
    assert info.cpu().numpy().tolist() == [0] * batch
    return w.cpu().numpy(), from_dev_colmajor(VR)
