"""A call whose device allocation fails returns LEO2D_ERR_ALLOC and leaves the handle as it
was, or without what it could not replace: the next calls either give what a fresh handle
gives, bit for bit, or refuse.  Failures are forced from the host: allocations above
LEO2D_ALLOC_LIMIT bytes fail, at limits that stop a call at its first and at later buffers."""
import os

import numpy as np
import pytest

from conftest import ROOT

import leo2d_amd as L
from leo2d_amd import workloads as W

pytestmark = pytest.mark.gpu


class _Limit:
    """Allocations above `most` bytes fail inside the block, which has to end in ERR_ALLOC."""

    def __init__(self, monkeypatch, most):
        self.mp, self.most = monkeypatch, most

    def __enter__(self):
        self.mp.setenv("LEO2D_ALLOC_LIMIT", str(self.most))

    def __exit__(self, kind, err, tb):
        self.mp.delenv("LEO2D_ALLOC_LIMIT")
        assert kind is L.Leo2dError and err.code == L.ERR_ALLOC, (kind, err)
        return True


# 600 rows of 40 -> 2 x 96 -> 200: bf16 inputs 48,000 bytes, FP32 inputs 96,000, outputs 480,000,
# pre-activations 230,400
@pytest.mark.parametrize("most", [1000, 50_000, 100_000, 300_000])
def test_network_after_a_failed_allocation(monkeypatch, most):
    rng = np.random.default_rng(0)
    x = rng.standard_normal((600, 40)).astype(np.float32)
    t = rng.standard_normal((600, 200)).astype(np.float32)
    fresh = L.Mlp(0, 40, 96, 2, 200, seed=1)
    loss, grad = fresh.gradients(x, t)
    few = fresh.forward(x[:100])
    fresh.close()
    net = L.Mlp(0, 40, 96, 2, 200, seed=1)
    assert np.array_equal(net.forward(x[:100]), few)
    for _ in range(2):
        with _Limit(monkeypatch, most):
            net.gradients(x, t)
        assert np.array_equal(net.forward(x[:100]), few)
        with _Limit(monkeypatch, most):
            L.mlp_ensemble([net], x)
        got = net.gradients(x[:100], t[:100])
        assert np.isfinite(got[0])
    assert net.gradients(x, t)[0] == loss and np.array_equal(net.gradients(x, t)[1], grad)
    net.close()


def _matrix(n, seed, half=3):
    """Symmetric band of 2 half + 1 entries a row, spectrum inside [-1, 1]."""
    rng = np.random.default_rng(seed)
    A = np.zeros((n, n))
    for k in range(1, half + 1):
        i = np.arange(n - k)
        A[i, i + k] = A[i + k, i] = rng.uniform(-1, 1, n - k)
    A /= 1.01 * np.max(np.abs(A).sum(axis=1))
    mask = A != 0
    rp = np.concatenate([[0], np.cumsum(mask.sum(axis=1))]).astype(np.int64)
    return rp, np.nonzero(mask)[1].astype(np.int32), A[mask]


# 900 rows of 6 entries: row pointers 7,208 bytes, columns 21,612, values 43,224
@pytest.mark.parametrize("most", [1000, 10_000, 30_000])
def test_upload_after_a_failed_allocation(monkeypatch, most):
    """The handle holds no Hamiltonian (300 rows with other rows' pointers would read past
    it) until the next upload; a batch keeps the one appended before."""
    dev = L.Device(0)
    small, large = _matrix(300, 1), _matrix(900, 2)
    t = np.array([0, 5, 299])
    dev.csr_upload(*small)
    ref = dev.kpm(32, targets=t)
    dev.batch_append()
    bref = dev.batch_kpm(32, 4, seed=1)
    for _ in range(2):
        with _Limit(monkeypatch, most):
            dev.csr_upload(*large)
        for call in (dev.csr_info, dev.csr_copy, dev.spectral_bounds, dev.batch_append, lambda: dev.kpm(32, targets=t),
                     lambda: dev.kpm(32, targets=t, noalloc=True)):
            with pytest.raises(L.Leo2dError) as e:
                call()
            assert e.value.code == L.ERR_STATE
        assert np.array_equal(dev.batch_kpm(32, 4, seed=1), bref)
        dev.csr_upload(*small)
        assert np.array_equal(dev.kpm(32, targets=t), ref)
    dev.csr_upload(*large)
    assert dev.csr_info()[0] == 900
    dev.close()


def _jobs(dev, sizes):
    for k, n in enumerate(sizes):
        dev.csr_upload(*_matrix(n, 10 + k))
        dev.batch_append()


# stacked: 5,000 rows, 40,008 bytes of row pointers, 29,976 entries, 119,968 bytes of columns, 239,872 of values
@pytest.mark.parametrize("most", [1000, 50_000, 150_000])
def test_stack_after_a_failed_allocation(monkeypatch, most):
    """Jobs appended after a run stay pending until their stack is whole."""
    fresh = L.Device(0)
    _jobs(fresh, (2000, 3000))
    ref = fresh.batch_kpm(32, 4, seed=1)
    fresh.close()
    dev = L.Device(0)
    _jobs(dev, (2000,))
    for graph in (False, True):
        first = dev.batch_kpm(32, 4, seed=1, graph=graph)
        assert np.array_equal(first[0], ref[0])
    dev.csr_upload(*_matrix(3000, 11))
    dev.batch_append()
    info = dev.batch_info()
    for _ in range(2):
        with _Limit(monkeypatch, most):
            dev.batch_kpm(32, 4, seed=1)
        assert dev.batch_info() == info == (2, 5000, info[2])
    for graph in (False, True, True):
        assert np.array_equal(dev.batch_kpm(32, 4, seed=1, graph=graph), ref)
    dev.close()


@pytest.mark.parametrize("mode", [L.BATCH_ROW_GROUPS, L.BATCH_ENTRY_SLOTS])
def test_batch_tiles_after_a_failed_allocation(monkeypatch, mode):
    """125 tiles of 16 rows are 504 bytes of first rows, 16 of 128 rows 68."""
    dev = L.Device(0)
    _jobs(dev, (2000,))
    ref = dev.batch_kpm(32, 4, seed=1, mode=mode, tile_rows=128)
    for graph in (False, True):
        with _Limit(monkeypatch, 400):
            dev.batch_kpm(32, 4, seed=1, mode=mode, tile_rows=16, graph=graph)
        assert np.array_equal(dev.batch_kpm(32, 4, seed=1, mode=mode, tile_rows=128, graph=graph), ref)
    dev.close()


def _state_error(*calls):
    for call in calls:
        with pytest.raises(L.Leo2dError) as e:
            call()
        assert e.value.code == L.ERR_STATE


# 944 orbitals: grid indices 15,104 bytes, positions 22,656, orders 3,776
@pytest.mark.parametrize("most", [100, 10_000, 20_000])
def test_geometry_after_a_failed_allocation(monkeypatch, most):
    """No geometry until every array is there: another one's pairs would be searched on
    arrays that are gone."""
    old, new = (L.Geometry(L.Deck(W.tblg_flake_deck(3.0, r, M=16))) for r in (8.0, 20.0))
    dev = L.Device(0)
    dev.set_geometry(new)
    dev.assemble(new.jobs()[0], L.PATTERN_PRUNED)
    ref = dev.csr_copy()
    dev.set_geometry(old)
    dev.assemble(old.jobs()[0], L.PATTERN_PRUNED)
    with _Limit(monkeypatch, most):
        dev.set_geometry(new)
    _state_error(dev.pairs_build, lambda: dev.assemble(new.jobs()[0], L.PATTERN_PRUNED), dev.csr_info)
    dev.set_geometry(new)
    dev.assemble(new.jobs()[0], L.PATTERN_PRUNED)
    assert all(np.array_equal(a, b) for a, b in zip(dev.csr_copy(), ref))
    dev.close()


@pytest.mark.parametrize("most", [100, 5_000, 10_000])
def test_pairs_after_a_failed_allocation(monkeypatch, most):
    """944 orbitals: counts of 3,776 and 7,552 bytes, lists above; the next assembly searches
    the pairs again."""
    geom = L.Geometry(L.Deck(W.tblg_flake_deck(3.0, 20.0, M=16)))
    dev = L.Device(0)
    dev.set_geometry(geom)
    dev.assemble(geom.jobs()[0], L.PATTERN_PRUNED)
    ref = dev.csr_copy()
    with _Limit(monkeypatch, most):
        dev.pairs_build()
    _state_error(dev.pairs_method)
    dev.assemble(geom.jobs()[0], L.PATTERN_PRUNED)
    assert all(np.array_equal(a, b) for a, b in zip(dev.csr_copy(), ref))
    dev.close()


def test_relaxation_after_a_failed_allocation(monkeypatch):
    geom = L.Geometry(L.Deck(open(os.path.join(ROOT, "tests", "decks", "tblg_relax_cell.in")).read()))
    job = geom.jobs()[0]
    job.strain_type = 1
    c = 1e-3 * np.random.default_rng(0).standard_normal((3, 4))   # max_k = 2: four coefficients a component
    dev = L.Device(0)
    dev.set_geometry(geom)
    dev.set_relaxation(2, c)
    dev.assemble(job, L.PATTERN_PRUNED)
    ref = dev.csr_copy()
    with _Limit(monkeypatch, 50):
        dev.set_relaxation(2, c)
    _state_error(lambda: dev.assemble(job, L.PATTERN_PRUNED))
    dev.set_relaxation(2, c)
    dev.assemble(job, L.PATTERN_PRUNED)
    assert all(np.array_equal(a, b) for a, b in zip(dev.csr_copy(), ref))
    dev.close()
