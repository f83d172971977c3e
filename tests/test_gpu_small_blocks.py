"""Blocks of 1 to 8 vectors (lanes grouped on a row) and the deferred moment
reductions, on random Hermitian matrices whose rows end at the edges of a lane
group's rounds: empty rows, rows of 1, 2, 3, 16, 47, 48, 49 and 200 entries, the
last row among them, so that the wide entry loads reach the arrays' end.
Against a dense FP64 recursion; 1e-12 mu_0 as in test_gpu_parity.py (the sums
run in another order)."""
import numpy as np
import pytest
import scipy.sparse as sp

import leo2d_amd as L

pytestmark = pytest.mark.gpu


def _matrix(n, rng, cpx, longest):
    """Symmetric pattern with row lengths spread over 0 .. longest; spectrum inside [-1, 1]."""
    A = np.zeros((n, n), dtype=complex if cpx else float)
    want = [1, 2, 3, 16, 47, 48, 49, longest]
    for i in range(1, n - 1, 3):
        for j in rng.choice(n, size=min(n, want[(i // 3) % len(want)]) // 2, replace=False):
            if j != 0:
                v = rng.standard_normal() + (1j * rng.standard_normal() if cpx else 0)
                A[i, j] = v
                A[j, i] = np.conj(v)
    A[n - 1, n - 1] = 0.5
    A[np.arange(n), np.arange(n)] = A.diagonal().real
    A /= 1.01 * max(1.0, np.max(np.abs(A).sum(axis=1)))
    mask = A != 0
    rp = np.concatenate([[0], np.cumsum(mask.sum(axis=1))]).astype(np.int64)
    ci = np.nonzero(mask)[1].astype(np.int32)
    return A, rp, ci, A[mask]


def _moments(A, V, M):
    """<v|T_n|v> of the columns of V."""
    a, b = V, A @ V
    mu = [np.sum(np.abs(V) ** 2, axis=0), np.sum(np.conj(V) * b, axis=0).real]
    for _ in range(2, M):
        a, b = b, 2 * (A @ b) - a
        mu.append(np.sum(np.conj(V) * b, axis=0).real)
    return np.array(mu).T


@pytest.mark.parametrize("cpx", [False, True])
@pytest.mark.parametrize("n,longest", [(1, 1), (17, 12), (400, 200), (700, 700)])
@pytest.mark.parametrize("R", [1, 2, 3, 4, 8])
def test_small_blocks(cpx, n, longest, R):
    rng = np.random.default_rng(n + R)
    A, rp, ci, v = _matrix(n, rng, cpx, longest)
    dev = L.Device(0)
    dev.csr_upload(rp, ci, v.astype(complex) if cpx else v)
    M = 64
    t = rng.integers(0, n, R).astype(np.int32)
    E = np.zeros((n, R))
    E[t, np.arange(R)] = 1.0
    ref = _moments(A, E, M)
    for scheme in (L.SCHEME_REFERENCE, L.SCHEME_DOUBLING):
        mu = dev.kpm(M, targets=t, scheme=scheme)
        assert dev.timing().kernel == 2
        assert np.max(np.abs(mu - ref)) <= 1e-12
    X = rng.standard_normal((R, n)) + 1j * rng.standard_normal((R, n))
    refx = _moments(A, X.T, M)
    mux = dev.kpm(M, vectors=X)
    assert np.max(np.abs(mux - refx)) <= 1e-12 * np.max(refx[:, 0])
    assert np.array_equal(mu, dev.kpm(M, targets=t, scheme=L.SCHEME_DOUBLING, noalloc=True))
    dev.close()


@pytest.mark.parametrize("R", [4, 8])
@pytest.mark.parametrize("cpx", [False, True])
def test_small_batch_blocks(R, cpx):
    """Stacked jobs of 1, 33 and 260 rows: tiles of fewer rows than a round, and more."""
    rng = np.random.default_rng(R)
    dev = L.Device(0)
    mats, targets = [], []
    for n in (1, 33, 260):
        A, rp, ci, v = _matrix(n, rng, cpx, min(n, 100))
        dev.csr_upload(rp, ci, v.astype(complex) if cpx else v)
        dev.batch_append()
        mats.append(A)
        targets.append(rng.integers(0, n, R))
    for graph in (False, True):
        mu = dev.batch_kpm(48, R, targets=np.array(targets), graph=graph)
        for A, t, m in zip(mats, targets, mu):
            E = np.zeros((A.shape[0], R))
            E[t, np.arange(R)] = 1.0
            assert np.max(np.abs(m - _moments(A, E, 48))) <= 1e-12
    dev.close()


def _band(n, half, cpx, rng):
    """Hermitian band of 2 half + 1 entries a row (fewer at its ends), spectrum inside [-1, 1]."""
    d = {0: rng.standard_normal(n)}
    for k in range(1, half + 1):
        v = rng.standard_normal(n - k) + (1j * rng.standard_normal(n - k) if cpx else 0)
        d[k], d[-k] = v, np.conj(v)
    A = sp.diags(list(d.values()), list(d.keys()), format="csr")
    A = A / (1.01 * np.max(abs(A).sum(axis=1)))
    A.sort_indices()
    return A.indptr.astype(np.int64), A.indices.astype(np.int32), A.data, A


# either side of each line of the choice between lanes per row (2) and a lane per vector (0), and of
# 16 against 64 lanes per row: rows, half band, complex H, vectors, kernel
@pytest.mark.parametrize("n,half,cpx,R,kernel", [
    (4095, 15, False, 8, 2), (4096, 15, False, 8, 0), (4097, 15, True, 5, 0), (8191, 40, True, 8, 2),
    (8191, 40, False, 8, 0), (8192, 50, True, 8, 0), (16383, 15, True, 4, 2), (16384, 15, True, 3, 0),
    (16384, 50, False, 4, 2), (131072, 2, False, 4, 0), (131073, 2, True, 4, 2), (131073, 2, False, 2, 2),
    (8191, 33, False, 2, 2), (8192, 33, True, 1, 2), (8193, 50, False, 2, 2)])
def test_few_vectors_on_many_rows(n, half, cpx, R, kernel):
    """Complex vectors, FP64, against the same recursion in numpy; 1e-12 mu_0 as above."""
    rng = np.random.default_rng(n + half)
    rp, ci, v, A = _band(n, half, cpx, rng)
    X = rng.standard_normal((R, n)) + 1j * rng.standard_normal((R, n))
    dev = L.Device(0)
    dev.csr_upload(rp, ci, v)
    M = 16
    ref = _moments(A, X.T, M)
    print("case", n, half, cpx, R, flush=True)
    mu = dev.kpm(M, vectors=X)
    assert dev.timing().kernel == kernel
    assert np.max(np.abs(mu - ref)) <= 1e-12 * np.max(ref[:, 0])
    if 2 * n * 16 * 8 < 30_000_000:
        assert np.array_equal(mu, dev.kpm(M, vectors=X, noalloc=True))
    dev.close()
