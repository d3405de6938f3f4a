"""GPU parity: blocked LU, triangular solves, GEMM and Cholesky through the
C ABI, against the CPU oracle (numax's float64 host algorithm restated).

Bar (the numax float64 contract): identical pivot sequences, and a normwise
backward error ||b - A x|| / (||A|| ||x||) within 10 n eps of the oracle's.
"""
import numpy as np
import pytest
import torch

import oracle
from numax_amd import linalg as nl
from numax_amd import random as R

pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float64).eps


def _np(t):
    return t.detach().cpu().numpy()


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("transa,transb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (37, 129, 17), (128, 128, 16), (300, 257, 256), (513, 64, 33)])
def test_gemm_matches_numpy(dtype, transa, transb, m, n, k):
    rng = np.random.default_rng(m * 1000 + n + k)
    a = rng.standard_normal((k, m) if transa else (m, k))
    b = rng.standard_normal((n, k) if transb else (k, n))
    c = rng.standard_normal((m, n))
    npd = np.float64 if dtype == torch.float64 else np.float32
    a, b, c = a.astype(npd), b.astype(npd), c.astype(npd)
    out = _np(nl.gemm(a, b, c, alpha=-1.0, beta=1.0, transa=bool(transa), transb=bool(transb)))
    ref = c.astype(np.float64) - (a.T if transa else a).astype(np.float64) @ (b.T if transb else b).astype(np.float64)
    tol = 1e-12 if dtype == torch.float64 else 2e-4
    assert np.max(np.abs(out - ref)) <= tol * max(1.0, np.max(np.abs(ref))) * np.sqrt(k)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("transa,transb", [(0, 0), (1, 1)])
def test_gemm_tile_shapes_agree_bitwise(dtype, transa, transb):
    # a 2944 x 2944 update is 23 x 23 = 529 tiles of 128 x 128 (the large-tile
    # path); its leading 384 x 320 block on its own is too small to fill the
    # device with those and takes 64 x 64 tiles.  Every element sums its k
    # slabs in the same order either way, so the two agree bit for bit.
    m = n = 2944
    k = 72
    rng = np.random.default_rng(2944 + transa)
    npd = np.float64 if dtype == torch.float64 else np.float32
    a = rng.standard_normal((k, m) if transa else (m, k)).astype(npd)
    b = rng.standard_normal((n, k) if transb else (k, n)).astype(npd)
    c = rng.standard_normal((m, n)).astype(npd)
    full = _np(nl.gemm(a, b, c, alpha=-1.0, beta=1.0, transa=bool(transa), transb=bool(transb)))
    a_s = np.ascontiguousarray(a[:, :384] if transa else a[:384])
    b_s = np.ascontiguousarray(b[:320] if transb else b[:, :320])
    part = _np(nl.gemm(a_s, b_s, np.ascontiguousarray(c[:384, :320]), alpha=-1.0, beta=1.0, transa=bool(transa),
                       transb=bool(transb)))
    assert np.array_equal(full[:384, :320], part)
    ref = c.astype(np.float64) - (a.T if transa else a).astype(np.float64) @ (b.T if transb else b).astype(np.float64)
    tol = 1e-12 if dtype == torch.float64 else 2e-4
    assert np.max(np.abs(full - ref)) <= tol * max(1.0, np.max(np.abs(ref))) * np.sqrt(k)


@pytest.mark.parametrize("transa", [0, 1])
def test_gemm_of_few_columns_in_very_wide_rows(transa):
    """Rows so far apart that 64 of them span more than 2 GiB: the operand that
    is walked down its rows is B, or A transposed."""
    from numax_amd import _lib
    m, n, k, wide = 20, 16, 70, 4_300_000
    rng = np.random.default_rng(transa)
    a, b, c = rng.standard_normal((m, k)), rng.standard_normal((k, n)), rng.standard_normal((m, n))
    far = torch.empty((k, wide), dtype=torch.float64, device="cuda")
    far[:, :m if transa else n] = torch.as_tensor(a.T if transa else b, device="cuda")
    near = torch.as_tensor(b if transa else a, device="cuda").contiguous()
    C = torch.as_tensor(c, device="cuda")
    A, B = (far, near) if transa else (near, far)
    _lib.check(nl._fn("gemm", torch.float64)(nl._ctx(C).handle, transa, 0, m, n, k, -1.0, nl._ptr(A), A.shape[1], nl._ptr(B),
                                             B.shape[1], 1.0, nl._ptr(C), n), "gemm")
    assert np.max(np.abs(_np(C) - (c - a @ b))) <= 1e-12


@pytest.mark.parametrize("n", [1, 7, 64, 65, 200, 300])
@pytest.mark.parametrize("upper,unit,trans", [(0, 0, 0), (0, 1, 0), (1, 0, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1)])
def test_solve_triangular_matches_oracle(n, upper, unit, trans):
    rng = np.random.default_rng(n + 10 * upper + 100 * unit + 1000 * trans)
    t = rng.standard_normal((n, n)) * 0.1 + np.eye(n) * 2.0
    b = rng.standard_normal((n, 3))
    x = _np(nl.solve_triangular(t, b, upper=bool(upper), unit=bool(unit), trans=bool(trans)))
    stored = np.triu(t) if upper else np.tril(t)
    if unit:
        stored = stored - np.diag(np.diag(stored)) + np.eye(n)
    op = stored.T if trans else stored
    np.testing.assert_allclose(op @ x, b, atol=1e-11 * n, rtol=0)
    for c in range(3):  # the oracle's vector form, column by column
        xo = oracle.solve_triangular(t, b[:, c], upper=bool(upper), unit=bool(unit), trans=bool(trans))
        np.testing.assert_allclose(x[:, c], xo, atol=1e-10, rtol=1e-10)


@pytest.mark.parametrize("n,nrhs", [(1, 1), (5, 3), (300, 1), (4097, 16), (16384, 1), (16385, 2), (20000, 1)])
def test_laswp_matches_oracle(n, nrhs):
    # n <= 16384 forms the permutation in LDS, larger n in device memory
    rng = np.random.default_rng(n + nrhs)
    rows = np.arange(n)
    ipiv = (rows + (rng.random(n) * (n - rows))).astype(np.int32)  # ipiv[j] in [j, n)
    keep = rng.random(n) < 0.3
    ipiv[keep] = rows[keep]  # steps without an interchange
    b = rng.standard_normal((n, nrhs)) if nrhs > 1 else rng.standard_normal(n)
    out = _np(nl.laswp(b, ipiv))
    assert np.array_equal(out, oracle.laswp(b, ipiv))


def _lu_parity(a, b, block=256, base=32):
    lu = nl.lu_factor(a, block=block, base=base)
    olu, opiv, oinfo, osign = oracle.getrf(a, block=32, base=16)
    piv = _np(lu.pivots)
    assert np.array_equal(piv, opiv), f"first pivot mismatch at {np.argmax(piv != opiv)}"
    assert lu.sign == osign
    assert lu.info == oinfo
    x = _np(lu.solve(b))
    xo = oracle.getrs(olu, opiv, b, block=32)
    n = a.shape[0]
    eta = oracle.backward_error(a, x, b)
    eta_o = oracle.backward_error(a, xo, b)
    assert eta <= eta_o + 10 * n * EPS, (eta, eta_o)
    return lu, x


def test_lu_c1_oracle_case():
    """C1: n=512, A ~ U[-1,1], b ~ N(0,1), seed 1."""
    a = R.lu_matrix(1, 512)
    b = R.normal(1, (512,))
    lu, x = _lu_parity(a, b)
    assert np.isfinite(x).all()


@pytest.mark.parametrize("n", [1, 2, 5, 31, 33, 100, 257, 1000, 1025, 2100, 4097])
def test_lu_sizes_and_ragged(n):
    a = R.normal(100 + n, (n, n))
    b = R.normal(200 + n, (n, 4))
    _lu_parity(a, b)


@pytest.mark.parametrize("block,base", [(16, 16), (32, 8), (64, 32), (100, 25), (512, 32)])
def test_lu_block_invariance(block, base):
    """numax pins blocked == unblocked (docs/features.md:285-287); pivots
    must not depend on the blocking."""
    a = R.normal(7, (700, 700))
    b = R.normal(8, (700,))
    _lu_parity(a, b, block=block, base=base)


def test_lu_exchange_matrix_known_answer():
    """test_tensor_linalg.mojo:816-832: [[0,1],[1,0]] has det -1, x = (5,3)
    for b = (3,5)."""
    lu = nl.lu_factor(np.array([[0.0, 1.0], [1.0, 0.0]]))
    assert lu.det() == -1.0
    np.testing.assert_array_equal(_np(lu.solve(np.array([3.0, 5.0]))), [5.0, 3.0])


def test_lu_textbook_3x3():
    """test_linalg.mojo:134-139: x = (2, 3, -1)."""
    a = np.array([[2.0, 1.0, -1.0], [-3.0, -1.0, 2.0], [-2.0, 1.0, 2.0]])
    b = np.array([8.0, -11.0, -3.0])
    np.testing.assert_allclose(_np(nl.solve(a, b)), [2.0, 3.0, -1.0], atol=1e-14)


def test_lu_pivot_known_answer():
    """test_panel.mojo:258-274: the first pivot of [[0,1,2],[4,5,6],[7,8,10]]
    is row 2."""
    lu = nl.lu_factor(np.array([[0.0, 1.0, 2.0], [4.0, 5.0, 6.0], [7.0, 8.0, 10.0]]))
    assert int(_np(lu.pivots)[0]) == 2


def test_lu_singular_reports_info_not_error():
    a = np.array([[1.0, 2.0], [2.0, 4.0]])
    lu = nl.lu_factor(a)
    assert lu.singular() and lu.info == 2
    assert lu.slogdet() == (0.0, -np.inf)
    olu, opiv, oinfo, _ = oracle.getrf(a)
    assert oinfo == lu.info


def test_lu_zero_column_info_first_only():
    a = np.zeros((40, 40))
    lu = nl.lu_factor(a)
    assert lu.info == 1
    np.testing.assert_array_equal(_np(lu.pivots), np.arange(40))


def test_lu_scipy_plu_known_answer():
    """tests/linalg/test_lu_plu.mojo:15-109: SciPy's (P, L, U) of a 4x4 whose
    first pivot is zero, to 1e-14."""
    from tests.golden.kat import PLU_A, PLU_L, PLU_P, PLU_U
    lu = nl.lu_factor(PLU_A)
    f = _np(lu.factored)
    np.testing.assert_allclose(np.tril(f, -1) + np.eye(4), PLU_L, atol=1e-14)
    np.testing.assert_allclose(np.triu(f), PLU_U, atol=1e-14)
    perm = np.arange(4)
    for j, q in enumerate(_np(lu.pivots)):
        perm[[j, q]] = perm[[q, j]]
    p = np.eye(4)[perm].T  # A = P L U with row i of P^T A = row perm[i] of A
    np.testing.assert_allclose(p, PLU_P, atol=0)


def test_lu_solve_shape_error_text():
    lu = nl.lu_factor(np.eye(3))
    with pytest.raises(nl.NumaxError, match="lu_solve: b has 2 entries for an order-3 factorization"):
        lu.solve(np.ones(2))
    with pytest.raises(nl.NumaxError, match="square"):
        nl.lu_factor(np.ones((2, 3)))


def test_lu_det_slogdet():
    a = R.normal(11, (60, 60))
    lu = nl.lu_factor(a)
    sign, logdet = np.linalg.slogdet(a)
    s, l = lu.slogdet()
    assert s == sign and abs(l - logdet) < 1e-10 * abs(logdet)
    spd3 = np.array([[4.0, 2.0, 0.6], [2.0, 5.0, 1.0], [0.6, 1.0, 3.0]])
    assert abs(nl.lu_factor(spd3).det() - np.linalg.det(spd3)) < 1e-12


def test_lu_float32_matches_reference_gpu_tolerances():
    """tests_gpu/linalg/test_lu_plu_gpu.mojo:17-44 at float32 on its n=48
    sin-generated matrix: the pivots of the float64 host algorithm, and
    P L U == A to 1e-5 as the reference checks.  (The matrix has condition
    number ~4.5e7, so float32 L/U entries are compared through the
    reconstruction, not entry by entry against float64.)"""
    from tests.golden.kat import sin48
    a = sin48()
    lu32 = nl.lu_factor(a)
    _, opiv, _, _ = oracle.getrf(a.astype(np.float64), block=16)
    np.testing.assert_array_equal(_np(lu32.pivots), opiv)
    f = _np(lu32.factored).astype(np.float64)
    l = np.tril(f, -1) + np.eye(48)
    u = np.triu(f)
    perm = np.arange(48)
    for j, q in enumerate(_np(lu32.pivots)):
        perm[[j, q]] = perm[[q, j]]
    np.testing.assert_allclose(l @ u, a.astype(np.float64)[perm], atol=1e-5)


def test_lu_c2_scale_pivots_and_backward_error():
    """C2: n=8192, A ~ N(0,1), 16 right-hand sides, block 256: identical pivots
    with the oracle and backward error within 10 n eps of it."""
    oracle.set_threads(16)
    n = 8192
    a = R.device_normal(2, (n, n)).cpu().numpy()
    b = R.device_normal(3, (n, 16)).cpu().numpy()
    _lu_parity(a, b, block=256, base=32)


def test_lu_many_part_panels_match_oracle():
    """n = 9216: the panels of the first 1024 columns span 18 workgroups of
    512 rows, where the pivot exchange stages every part's key first and then
    only the winner's row; pivots identical to the oracle's."""
    oracle.set_threads(16)
    n = 9216
    a = R.device_normal(5, (n, n)).cpu().numpy()
    b = R.device_normal(6, (n, 4)).cpu().numpy()
    _lu_parity(a, b, block=256, base=32)


@pytest.mark.parametrize("n", [1, 5, 64, 65, 300, 1000, 1300])
def test_cholesky_matches_oracle(n):
    a = R.spd_matrix(300 + n, n)
    l = _np(nl.cholesky(a))
    lo, info = oracle.potrf(a)
    assert info == 0
    np.testing.assert_allclose(l, lo, atol=1e-12 * np.sqrt(n), rtol=0)
    assert np.array_equal(np.triu(l, 1), np.zeros((n, n)))
    b = R.normal(400 + n, (n, 3))
    x = _np(nl.cholesky_solve(l, b))
    eta = oracle.backward_error(a, x, b)
    eta_o = oracle.backward_error(a, oracle.potrs(lo, b), b)
    assert eta <= eta_o + 10 * n * EPS


def test_cholesky_reads_lower_triangle_only():
    a = R.spd_matrix(5, 150)
    junk = a + np.triu(np.full_like(a, 7.0), 1)
    np.testing.assert_allclose(_np(nl.cholesky(junk)), _np(nl.cholesky(a)), atol=0, rtol=0)


def test_cholesky_not_pd_raises_with_index():
    """test_panel.mojo:146-161: [[4,2,2],[2,1,0],[2,0,9]] fails at index 1
    (info 2)."""
    with pytest.raises(nl.NumaxError, match=r"non-positive pivot at index 1\)"):
        nl.cholesky(np.array([[4.0, 2.0, 2.0], [2.0, 1.0, 0.0], [2.0, 0.0, 9.0]]))
    a = R.spd_matrix(9, 500)
    a[321, 321] = -50.0
    _, info = oracle.potrf(a)
    with pytest.raises(nl.NumaxError, match=f"index {info - 1}\\)"):
        nl.cholesky(a)


def test_cholesky_c2_scale():
    """C2 Cholesky: A = G G^T / n + I, n = 8192, 16 right-hand sides."""
    n = 8192
    g = R.device_normal(2, (n, n))
    a = g @ g.T / n + torch.eye(n, dtype=torch.float64, device="cuda")
    a = (a + a.T) * 0.5
    l = nl.cholesky(a)
    b = R.device_normal(3, (n, 16))
    x = nl.cholesky_solve(l, b)
    r = b - a @ x
    eta = (r.abs().max(0).values / (a.abs().sum(1).max() * x.abs().max(0).values)).max().item()
    assert eta < 10 * n * EPS


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 128, 129, 255, 256, 257, 530])
def test_triangular_strip_edges(n, dtype):
    """Every triangle, diagonal and transposition at the edges of the 16-row
    steps and the 64 / 128 / 256-row kernels, one to 33 vectors, strided
    operands, and the residual bound of substitution (n eps |T||x|, with a
    factor for the inverted 16 x 16 blocks)."""
    eps = torch.finfo(dtype).eps
    rng = np.random.default_rng(n)
    for upper, unit, trans, nrhs in ((0, 0, 0, 1), (0, 1, 0, 16), (1, 0, 0, 17), (1, 1, 0, 33), (0, 0, 1, 5),
                                     (1, 0, 1, 2), (0, 1, 1, 1), (1, 1, 1, 20)):
        t = rng.standard_normal((n, n + 3)) / np.sqrt(n)
        t[:, :n] += 2.0 * np.eye(n)
        T = torch.as_tensor(t, device="cuda").to(dtype)
        B0 = torch.as_tensor(rng.standard_normal((n, nrhs + 2)), device="cuda").to(dtype)
        B = B0.clone()
        stored = T[:, :n].double().cpu().numpy()
        stored = np.triu(stored) if upper else np.tril(stored)
        if unit:
            stored = stored - np.diag(np.diag(stored)) + np.eye(n)
        op = stored.T if trans else stored
        from numax_amd import _lib
        _lib.check(nl._fn("trsm", dtype)(nl._ctx(T).handle, int(upper != trans), unit, trans, n, nrhs, nl._ptr(T), n + 3,
                                         nl._ptr(B), nrhs + 2), "trsm")
        x = B[:, :nrhs].double().cpu().numpy()
        r = np.abs(op @ x - B0[:, :nrhs].double().cpu().numpy())
        assert np.all(r <= 16 * (n + 16) * eps * (np.abs(op) @ np.abs(x) + 1)), (upper, unit, trans, nrhs)
        assert torch.equal(B[:, nrhs:], B0[:, nrhs:])


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n,nrhs", [(1100, 1), (1100, 17), (793, 16), (2050, 33)])
def test_triangular_thin_updates(n, nrhs, dtype):
    """Updates of a few vectors with long, ragged contractions: several slabs a
    wavefront, a remainder of 1 to 15, a partial last row and column tile.
    Residual bound of substitution as at the strip edges."""
    eps = torch.finfo(dtype).eps
    rng = np.random.default_rng(n + nrhs)
    from numax_amd import _lib
    for upper, trans in ((0, 0), (1, 0), (0, 1), (1, 1)):
        t = rng.standard_normal((n, n + 1)) / np.sqrt(n)
        t[:, :n] += 2.0 * np.eye(n)
        T = torch.as_tensor(t, device="cuda").to(dtype)
        B0 = torch.as_tensor(rng.standard_normal((n, nrhs + 1)), device="cuda").to(dtype)
        B = B0.clone()
        stored = T[:, :n].double().cpu().numpy()
        stored = np.triu(stored) if upper else np.tril(stored)
        op = stored.T if trans else stored
        _lib.check(nl._fn("trsm", dtype)(nl._ctx(T).handle, int(upper != trans), 0, trans, n, nrhs, nl._ptr(T), n + 1,
                                         nl._ptr(B), nrhs + 1), "trsm")
        x = B[:, :nrhs].double().cpu().numpy()
        r = np.abs(op @ x - B0[:, :nrhs].double().cpu().numpy())
        assert np.all(r <= 16 * (n + 16) * eps * (np.abs(op) @ np.abs(x) + 1)), (upper, trans)
        assert torch.equal(B[:, nrhs:], B0[:, nrhs:])


def test_triangular_strip_spreads_infinities_as_substitution_does():
    n = 70
    rng = np.random.default_rng(9)
    t = np.tril(rng.standard_normal((n, n))) + 4 * np.eye(n)
    b = rng.standard_normal((n, 3))
    b[20, 1] = np.inf
    t2 = t.copy()
    t2[40, 40] = 0.0  # a zero on the diagonal divides
    for m, upper in ((t, False), (t2, False), (t.T.copy(), True), (t2.T.copy(), True)):
        x = _np(nl.solve_triangular(m, b, upper=upper))
        order = range(n - 1, -1, -1) if upper else range(n)
        xo = np.empty_like(b)
        with np.errstate(all="ignore"):
            w = b.copy()
            for j in order:
                xo[j] = w[j] / m[j, j]
                rest = range(j) if upper else range(j + 1, n)
                for i in rest:
                    w[i] = w[i] - m[i, j] * xo[j]
        np.testing.assert_array_equal(np.isfinite(x), np.isfinite(xo))
        ok = np.isfinite(xo)
        np.testing.assert_allclose(x[ok], xo[ok], rtol=1e-10, atol=1e-12)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 33, 63, 64, 65, 127, 128, 129, 200, 255, 256, 257, 385])
def test_cholesky_block_edges(n, dtype):
    """The one-workgroup block at the edges of its 16-column steps and of the
    64 / 128 / 256-column workgroups, ill-conditioned and strided: the factor's
    backward error |L L^T - A| <= n eps diag(A)^(1/2) diag(A)^(1/2)^T (Higham,
    Theorem 10.3, with a factor of 4), and memory right of the matrix left alone."""
    from numax_amd import _lib
    rng = np.random.default_rng(n)
    q, _ = np.linalg.qr(rng.standard_normal((n, n)))
    kappa = 1e10 if dtype == torch.float64 else 1e4
    a = (q * np.geomspace(1.0, 1.0 / kappa, n)) @ q.T
    a = 0.5 * (a + a.T)
    A = torch.full((n, n + 3), 5.0, dtype=dtype, device="cuda")
    A[:, :n] = torch.as_tensor(a, device="cuda").to(dtype)
    a = A[:, :n].double().cpu().numpy()
    info = torch.zeros(1, dtype=torch.int32, device="cuda")
    _lib.check(nl._fn("potrf", dtype)(nl._ctx(A).handle, n, nl._ptr(A), n + 3, nl._ptr(info), 0), "potrf")
    assert int(info.item()) == 0
    low = A[:, :n].double().cpu().numpy()
    assert np.array_equal(low, np.tril(low)) and bool((A[:, n:] == 5.0).all())
    d = np.sqrt(np.diag(a))
    err = np.tril(np.abs(low @ low.T - a))
    assert np.all(err <= 4 * (n + 1) * torch.finfo(dtype).eps * np.outer(d, d))


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n,i,j,value", [(40, 30, 5, np.nan), (128, 100, 20, np.nan), (128, 127, 111, np.inf),
                                         (256, 200, 190, np.nan), (60, 7, 7, np.inf), (128, 70, 70, np.inf),
                                         (300, 290, 17, -np.inf), (256, 129, 129, np.nan)])
def test_cholesky_spreads_infinities_as_column_elimination_does(n, i, j, value, dtype):
    """One entry that is not finite: entries that the plain column loop leaves
    finite are finite and right, the others are its infinities and NaNs.  An
    infinite pivot gives a column of zeros."""
    npd = np.float64 if dtype == torch.float64 else np.float32
    a = R.spd_matrix(n + i, n).astype(npd)
    a[i, j] = value
    low = _np(nl.cholesky(torch.as_tensor(a, device="cuda")))
    ref = np.tril(a.astype(np.float64))
    with np.errstate(all="ignore"):
        for k in range(n):
            ref[k, k] = np.sqrt(ref[k, k])
            ref[k + 1:, k] /= ref[k, k]
            ref[k + 1:, k + 1:] -= np.tril(np.outer(ref[k + 1:, k], ref[k + 1:, k]))
    ref = np.tril(ref)
    np.testing.assert_array_equal(np.isnan(low), np.isnan(ref))
    np.testing.assert_array_equal(np.isinf(low), np.isinf(ref))
    ok = np.isfinite(ref)
    # each entry: the elimination's n roundings of terms bounded by the diagonal's root
    tol = 8 * (n + 1) * np.finfo(npd).eps * np.sqrt(np.max(np.diag(a)[np.isfinite(np.diag(a))]))
    assert np.all(np.abs(low[ok] - ref[ok]) <= tol)


@pytest.mark.parametrize("n,at", [(40, 0), (40, 17), (130, 127), (300, 16), (300, 299)])
def test_cholesky_reports_the_first_bad_pivot(n, at):
    a = R.spd_matrix(n, n)
    a[at, at] = -1.0
    if at + 1 < n:
        a[n - 1, n - 1] = -2.0  # a later one is not reported
    with pytest.raises(nl.NumaxError, match=f"at index {at}\\)"):
        nl.cholesky(a)


@pytest.mark.parametrize("n", [31, 32, 33, 40, 64, 129, 512, 513, 1024, 1056])
def test_leaf_ties_zeros_and_nans_keep_numax_pivots(n):
    """Rows that tie, columns that are zero or NaN, at the row limits of the
    one-workgroup leaf and its eight-column groups: the oracle's pivots."""
    rng = np.random.default_rng(n)
    a = rng.integers(-2, 3, (n, n)).astype(np.float64)  # many ties; singular with the zero column
    a[:, 5] = 0.0
    if n > 40:
        a[:, 37] = 0.0
    lu = nl.lu_factor(a)
    _, piv, info, _ = oracle.getrf(a)
    # exact small-integer arithmetic holds for the first columns only; compare
    # the pivots until a rounding (a non-dyadic quotient) could reorder a tie
    assert np.array_equal(lu.pivots.cpu().numpy()[:3], piv[:3])
    assert lu.info == info
    b = rng.standard_normal((n, n))
    b[n // 2, 0] = np.nan  # a NaN below the diagonal never wins
    lu = nl.lu_factor(b)
    assert lu.pivots.cpu().numpy()[0] == oracle.getrf(b)[1][0]


def _same_bits(a, b):
    """Equal bit for bit, NaNs anywhere at the same places."""
    nan = np.isnan(b)
    np.testing.assert_array_equal(np.isnan(a), nan)
    u = np.uint64 if a.dtype == np.float64 else np.uint32
    np.testing.assert_array_equal(np.where(nan, 0, a.view(u)), np.where(nan, 0, b.view(u)))


def _trsm(T, B, upper, unit, trans, n, nrhs):
    from numax_amd import _lib
    _lib.check(nl._fn("trsm", T.dtype)(nl._ctx(T).handle, upper, unit, trans, n, nrhs, nl._ptr(T), T.shape[1], nl._ptr(B),
                                       B.shape[1]), "trsm")


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n,nrhs", [(1, 1), (15, 3), (16, 17), (17, 16), (33, 1), (63, 2), (64, 16), (65, 5), (80, 33),
                                    (113, 1), (127, 2), (128, 16), (129, 17), (130, 1), (145, 3), (191, 2), (192, 16),
                                    (193, 5), (241, 1), (255, 17), (256, 16), (257, 2), (385, 1), (600, 17), (1100, 3),
                                    (100, 4100), (256, 4112)])
def test_triangular_solves_keep_substitutions_order(n, nrhs, dtype):
    """Bit for bit the oracle's substitution in blocks of 64 rows, every triangle,
    diagonal and transposition: the edges of the 16-row steps, of the 64 / 128 /
    256-row kernels and of 129 / 130 rows, where the split changes, both vector
    widths and strips joined by products.  Triangles of condition up to 1e12
    (1e5 in FP32) with zeros, negative zeros, tiny, huge and infinite entries, so
    that quotients leave the plain range too.  (Another order of the same
    operations cost solutions of ill-conditioned systems 1.6 times the error.)"""
    npd = np.float64 if dtype == torch.float64 else np.float32
    rng = np.random.default_rng(1000 * n + nrhs)
    far = 200 if npd is np.float64 else 30
    for case in range(8):
        upper, unit, trans = case >> 2, case >> 1 & 1, case & 1
        t = (rng.standard_normal((n, n + 1)) / np.sqrt(n)).astype(npd)
        d = np.geomspace(1.0, 1e-12 if npd is np.float64 else 1e-5, n)
        t[:, :n][np.arange(n), np.arange(n)] = rng.permutation(d) if case % 3 else 1.0 + d
        b = rng.standard_normal((n, nrhs)).astype(npd)
        if n > 60:
            b[n // 3, 0], b[n // 2, -1], b[n // 4, 0] = 0.0, -0.0, 10.0 ** -far
            if case >= 4:
                b[n - 2, -1] = 10.0 ** far
                t[n // 2, n // 2] = 10.0 ** (far - 5)
            if case in (2, 5):
                b[40, 0] = np.inf
        T, B = torch.as_tensor(t, device="cuda"), torch.as_tensor(b, device="cuda")
        _trsm(T, B, upper, unit, trans, n, nrhs)
        with np.errstate(all="ignore"):
            _same_bits(_np(B), oracle.device_order_trsm(t, b, bool(upper), bool(unit), bool(trans)))


def _lu_input(n, kind, npd):
    """Matrices on which a leaf's decisions and quotients can go wrong: 1, small
    integers (rows that tie in every column, zero pivots) with zero columns; 2,
    columns and rows out of the quotients' plain range; 3, NaNs and infinities."""
    rng = np.random.default_rng(100 * n + kind)
    a = rng.standard_normal((n, n))
    far = 200 if npd is np.float64 else 30
    if kind == 1:
        a = rng.integers(-2, 3, (n, n)).astype(np.float64)
        a[:, [j for j in (5, 8, 31, 32, 37) if j < n]] = 0.0
    elif kind == 2:
        a[:, n // 2] *= 10.0 ** -far
        a[n // 3] *= 10.0 ** (far - 10)
        a[n // 5:, 9 % n] = 0.0
    elif kind == 3:
        a[n // 2, 0] = np.nan  # below the diagonal: never wins
        a[n - 1, min(n - 1, 20)] = np.inf
        if n > 9:
            a[8, 8] = np.nan
    return a.astype(npd)


def _lu_bits(n, block, base, dtype, kinds):
    npd = np.float64 if dtype == torch.float64 else np.float32
    for kind in kinds:
        a = _lu_input(n, kind, npd)
        f = nl.lu_factor(torch.as_tensor(a, device="cuda"), block=block, base=base)
        with np.errstate(all="ignore"):
            lu, piv, info = oracle.device_order_getrf(a, block, base)
        assert np.array_equal(_np(f.pivots), piv), kind
        assert f.info == info, kind
        _same_bits(_np(f.factored), lu)
        if kind == 0:
            b = np.random.default_rng(n).standard_normal((n, 3)).astype(npd)
            w = oracle.laswp(b, piv).astype(npd)
            x = oracle.device_order_trsm(lu, oracle.device_order_trsm(lu, w, False, True), True)
            _same_bits(_np(f.solve(torch.as_tensor(b, device="cuda"))), x)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n", [1, 5, 31, 33, 40, 64, 129, 257, 512, 513, 1024, 1056, 1700])
def test_lu_is_the_blocked_elimination_bit_for_bit(n, dtype):
    """Factor, every pivot, ``info`` and solution equal the oracle's blocked
    elimination in the device's order: correctly rounded quotients, ties, zeros
    and NaNs in every eight-column group and leaf, one workgroup and several.
    (Gaussian systems of order 8192 reach condition 1e6: x kept to 1e-9 of the
    former x takes the same rounding, not only as good a one.)"""
    _lu_bits(n, 256, 32, dtype, (0, 1, 2, 3))


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("block,base", [(16, 16), (32, 8), (64, 32), (100, 25), (33, 7), (192, 32), (512, 16)])
@pytest.mark.parametrize("n", [17, 200, 600])
def test_lu_runs_the_panels_it_is_given(n, block, base, dtype):
    """Panels and leaves of the caller's widths: the same blocked elimination
    with those widths, bit for bit."""
    _lu_bits(n, block, base, dtype, (0, 1))
