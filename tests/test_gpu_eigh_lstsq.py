"""GPU parity of the batched Jacobi eigensolver and the batched tall-skinny
least squares against the FP64 oracle (numax's register-tier eigh,
numax/linalg/_array/eigen.mojo:316-392, and Householder lstsq,
numax/linalg/qr.mojo:746-821).

Bars (FP32 kernels, FP64 checks, tolerances stated here):
- eigh: sorted eigenvalues within 2e-5 * ||A||_2 of the oracle's and of
  LAPACK's; ||A V - V diag(w)|| <= 1e-4 ||A||, ||V^T V - I|| <= 1e-4; the
  closed form of the free-particle tridiagonal; trace and Frobenius identities.
- lstsq: x within 1e-4 relative of the FP64 oracle on well-conditioned
  Gaussian problems; the least-squares residual is orthogonal to range(A).
"""
import numpy as np
import pytest

import oracle
from numax_amd import linalg as nl

pytestmark = pytest.mark.gpu


def _pack(mats):
    n = np.array([m.shape[0] for m in mats], dtype=np.int32)
    oa = np.zeros(len(mats), dtype=np.int64)
    ow = np.zeros(len(mats), dtype=np.int64)
    oa[1:] = np.cumsum(n.astype(np.int64) ** 2)[:-1]
    ow[1:] = np.cumsum(n.astype(np.int64))[:-1]
    a = np.concatenate([m.astype(np.float32).ravel() for m in mats])
    return a, n, oa, ow


def _hamiltonian(n, omega):
    # finite-difference well on [-4, 4] (numax's quantum_well example, lines 66-80)
    h = 8.0 / (n - 1)
    x = np.linspace(-4.0, 4.0, n)
    a = np.diag(1.0 / h ** 2 + 0.5 * omega ** 2 * x ** 2)
    off = -0.5 / h ** 2
    a += np.diag(np.full(n - 1, off), 1) + np.diag(np.full(n - 1, off), -1)
    return a


def _mats(sizes, seed):
    rng = np.random.default_rng(seed)
    out = []
    for i, n in enumerate(sizes):
        if i % 2:
            out.append(_hamiltonian(n, rng.uniform(0.5, 2.0)))
        else:
            g = rng.standard_normal((n, n))
            out.append((g + g.T) / 2)
    return out


@pytest.mark.parametrize("sizes", [[1, 2, 3, 5, 8, 16, 24, 31, 32], [33, 40, 48, 63, 64], [24, 32, 48, 64] * 8])
def test_eigh_batched_matches_oracle(sizes):
    mats = _mats(sizes, seed=len(sizes))
    a, n, oa, ow = _pack(mats)
    w, v = nl.eigh_batched(a, n, oa, ow)
    w, v = w.cpu().numpy(), v.cpu().numpy()
    for p, m in enumerate(mats):
        k = m.shape[0]
        wp = w[ow[p]:ow[p] + k].astype(np.float64)
        vp = v[oa[p]:oa[p] + k * k].reshape(k, k).astype(np.float64)
        m32 = m.astype(np.float32).astype(np.float64)
        scale = max(np.abs(np.linalg.eigvalsh(m32)).max(), 1e-30)
        wo, _ = oracle.array_eigh(m32)
        assert np.max(np.abs(np.sort(wp) - np.sort(wo))) <= 2e-5 * scale, f"problem {p} n={k}"
        assert np.max(np.abs(np.sort(wp) - np.linalg.eigvalsh(m32))) <= 2e-5 * scale
        assert np.max(np.abs(m32 @ vp - vp * wp)) <= 1e-4 * scale
        assert np.max(np.abs(vp.T @ vp - np.eye(k))) <= 1e-4
        assert abs(wp.sum() - np.trace(m32)) <= 1e-4 * scale * k
        assert abs((wp ** 2).sum() - (m32 ** 2).sum()) <= 1e-4 * scale ** 2 * k


def test_eigh_free_particle_closed_form():
    # omega = 0: tridiagonal (-1/2h^2, 1/h^2, -1/2h^2), lambda_k = h^-2 (1 - cos(k pi / (n + 1)))
    mats = [_hamiltonian(n, 0.0) for n in (24, 32, 48, 64)]
    a, n, oa, ow = _pack(mats)
    w, _ = nl.eigh_batched(a, n, oa, ow, vectors=False)
    w = w.cpu().numpy()
    for p, m in enumerate(mats):
        k = m.shape[0]
        h = 8.0 / (k - 1)
        exact = (1.0 - np.cos(np.arange(1, k + 1) * np.pi / (k + 1))) / h ** 2
        assert np.max(np.abs(np.sort(w[ow[p]:ow[p] + k]) - exact)) <= 2e-5 * exact.max()


def test_eigh_ground_energy_quantum_well():
    # quantum_well.mojo:29-31: n = 24, omega = 1 ground energy ~ 0.496
    a, n, oa, ow = _pack([_hamiltonian(24, 1.0)])
    w, _ = nl.eigh_batched(a, n, oa, ow, vectors=False)
    assert abs(float(np.min(w.cpu().numpy()[:24])) - 0.496) < 0.01


@pytest.mark.parametrize("m,n,count", [(1024, 32, 64), (100, 7, 9), (32, 32, 3), (33, 1, 5)])
def test_lstsq_batched_matches_oracle(m, n, count):
    rng = np.random.default_rng(m + n)
    a = rng.standard_normal((count, m, n)).astype(np.float32)
    b = rng.standard_normal((count, m)).astype(np.float32)
    x = nl.lstsq_batched(a, b).cpu().numpy().astype(np.float64)
    for p in range(count):
        a64, b64 = a[p].astype(np.float64), b[p].astype(np.float64)
        xo = oracle.array_lstsq(a64, b64)
        assert np.max(np.abs(x[p] - xo)) <= 1e-4 * max(1.0, np.abs(xo).max()), f"problem {p}"
        r = b64 - a64 @ x[p]
        assert np.max(np.abs(a64.T @ r)) <= 1e-3 * np.linalg.norm(a64) * np.linalg.norm(b64)


@pytest.mark.parametrize("m,n", [(1, 1), (2, 2), (31, 16), (32, 17), (64, 16), (128, 32), (129, 31), (256, 15),
                                 (257, 32), (512, 8), (513, 17), (1024, 16), (1025, 32), (2048, 32), (2049, 5),
                                 (4032, 32), (4033, 31)])
def test_lstsq_batched_at_the_edges_of_its_row_and_column_tiles(m, n):
    """128 rows a wavefront, 1 to 16 wavefronts, 16-column register sets, and
    chunks of 2048 - 32 rows past 2048.  Backward stable, so the solution is
    within a few m n eps of exact for these well-conditioned problems."""
    count = 5
    rng = np.random.default_rng(1000 * m + n)
    a = rng.standard_normal((count, m, n))
    if m < 2 * n:  # square or nearly: keep the condition number small
        a[:, np.arange(n), np.arange(n)] += 2.0 * np.sqrt(m)
    a = a.astype(np.float32)
    b = rng.standard_normal((count, m)).astype(np.float32)
    a[3] = 0.0 if n == 1 else a[3]  # a zero column: non-finite, and only there
    x = nl.lstsq_batched(a, b).cpu().numpy().astype(np.float64)
    eps = np.finfo(np.float32).eps
    for p in range(count):
        if n == 1 and p == 3:
            assert not np.isfinite(x[p]).any()
            continue
        a64, b64 = a[p].astype(np.float64), b[p].astype(np.float64)
        xo = np.linalg.lstsq(a64, b64, rcond=None)[0]
        sv = np.linalg.svd(a64, compute_uv=False)
        kappa = sv[0] / sv[-1]
        bound = 4 * n * np.sqrt(m) * eps * kappa * (np.linalg.norm(b64) / sv[-1] + np.linalg.norm(xo))
        assert np.linalg.norm(x[p] - xo) <= bound, f"problem {p}"


def test_lstsq_tall_6x3_known_answer():
    from tests.golden import kat
    g = np.load(__import__("os").path.join(__import__("os").path.dirname(__file__), "golden", "goldens.npz"))
    b = np.array([1.0, -2.0, 3.0, 0.5, 4.0, -1.0])
    x = nl.lstsq_batched(kat.TALL_6x3[None].astype(np.float32), b[None].astype(np.float32)).cpu().numpy()[0]
    xo = oracle.array_lstsq(kat.TALL_6x3, b)
    assert np.allclose(x, xo, atol=1e-5, rtol=1e-5)
    assert "tall6x3_x" in g.files


def test_lstsq_shape_errors():
    with pytest.raises(nl.NumaxError):
        nl.lstsq_batched(np.zeros((2, 8, 4), np.float32), np.zeros((2, 7), np.float32))
    with pytest.raises(ValueError):
        nl.lstsq_batched(np.zeros((1, 8, 40), np.float32), np.zeros((1, 8), np.float32))


@pytest.mark.parametrize("sizes", [(31, 32), (5, 17, 32), (1, 2, 24), (33, 48, 64)])
def test_eigh_batched_keeps_non_finite_matrices_to_themselves(sizes):
    """A matrix with a NaN or an infinity beside every valid one: orders up to
    32 share a wavefront in pairs.  The valid ones come out as in a batch that
    holds no other, bit for bit."""
    rng = np.random.default_rng(sum(sizes))
    n = np.resize(np.array(sizes, dtype=np.int32), 240)
    mats = []
    for k in n:
        m = rng.standard_normal((k, k)).astype(np.float32)
        mats.append(m + m.T)
    offa, offw = np.zeros(len(n), dtype=np.int64), np.zeros(len(n), dtype=np.int64)
    offa[1:] = np.cumsum(n.astype(np.int64) ** 2)[:-1]
    offw[1:] = np.cumsum(n.astype(np.int64))[:-1]
    w0, v0 = (t.cpu().numpy() for t in nl.eigh_batched(np.concatenate([m.ravel() for m in mats]), n, offa, offw))
    bad = [p for p in range(len(n)) if p % 7 in (1, 3, 4)]
    for p in bad:
        i, j = rng.integers(0, n[p], 2)
        mats[p][i, j] = mats[p][j, i] = (np.nan, np.inf, -np.inf)[p % 3]
    w1, v1 = (t.cpu().numpy() for t in nl.eigh_batched(np.concatenate([m.ravel() for m in mats]), n, offa, offw))
    for p in range(len(n)):
        if p in bad:
            continue
        np.testing.assert_array_equal(w1[offw[p]:offw[p] + n[p]], w0[offw[p]:offw[p] + n[p]], err_msg=f"matrix {p}")
        np.testing.assert_array_equal(v1[offa[p]:offa[p] + n[p] ** 2], v0[offa[p]:offa[p] + n[p] ** 2], err_msg=f"matrix {p}")


@pytest.mark.parametrize("n", [1, 2, 3, 16, 17, 32])
@pytest.mark.parametrize("extra", [0, 1, 130, 2100])
def test_lstsq_batched_leaves_columns_that_are_zero_below_the_diagonal(n, extra):
    """Upper triangles over `extra` zero rows, as the last column of every square
    problem is one: no reflector squares the diagonal, so entries whose square
    under- or overflows solve like any other, a subnormal one too, and an
    infinity right of the diagonal reaches the unknowns above it only.  The
    solution is back substitution's, each unknown within n + 2 roundings of the
    terms it sums."""
    rng = np.random.default_rng(40 * n + extra)
    m, scales = n + extra, [1.0, 3e-30, 2e-23, 4e19, 2e37]
    a = np.zeros((len(scales) + 2, m, n), dtype=np.float32)
    b = rng.standard_normal((len(a), m)).astype(np.float32)
    for p, s in enumerate(scales + [1.0, 1.0]):
        a[p, :n] = (s * (np.triu(rng.uniform(-0.5, 0.5, (n, n)) / n, 1) + np.diag(rng.uniform(1.0, 2.0, n)))).astype(np.float32)
        b[p] *= np.float32(s)
    a[-1, n - 1, n - 1], b[-1, n - 1] = 3e-39, 1e-39
    if n > 2:
        a[-2, 0, n - 1] = np.inf
    x = nl.lstsq_batched(a, b).cpu().numpy().astype(np.float64)
    eps = np.finfo(np.float32).eps
    for p in range(len(a)):
        u, y = a[p, :n].astype(np.float64), b[p, :n].astype(np.float64)
        for i in range(n - 1, -1, -1):
            if not np.isfinite(u[i]).all():
                assert not np.isfinite(x[p, i])
                continue
            # against the unknowns that the kernel found, so that roundings do not add up
            terms = u[i, i + 1:] * x[p, i + 1:]
            bound = (n + 2) * eps * (np.abs(terms).sum() + abs(y[i])) / abs(u[i, i])
            assert abs(x[p, i] - (y[i] - terms.sum()) / u[i, i]) <= bound, (p, i)
