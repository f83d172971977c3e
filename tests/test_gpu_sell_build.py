"""Row tiles of the LDS-staged step where their layout on the device can go
wrong: matrices smaller than a tile, one row more than whole tiles, segments of
one tile and of several, tiles cut by the staged-row budget, rows too long for
the layout, which the CSR step runs, and the least rows it takes.  FP64 moments
within 1e-12 mu_0 of the oracle; the same tiles serve the FP32 recursion (2e-5
mu_0)."""
import numpy as np
import pytest

import leo2d_amd as L
from leo2d_amd import workloads as W

pytestmark = pytest.mark.gpu

# deck, orbitals, largest tile: the flakes leave remainders of 1 to 55 rows
CASES = {
    "one_tile": (W.tblg_flake_deck(5.0, 4.0, M=16), "56"),
    "two_tiles": (W.tblg_flake_deck(5.0, 6.5, M=16), "56"),
    "groups_cut": (W.tblg_flake_deck(5.0, 13.0, M=16), "5"),
    "short_segments": (W.tblg_flake_deck(5.0, 24.0, M=16), "56"),
    "long_segments": (W.tblg_flake_deck(5.0, 24.0, M=16), "4"),
}


@pytest.mark.parametrize("name", sorted(CASES))
@pytest.mark.parametrize("ucap", ["288", "70"])
def test_tiles_match_oracle(oracle_mod, monkeypatch, name, ucap):
    text, tmax = CASES[name]
    monkeypatch.setenv("LEO2D_KPM_VARIANT", "20")
    monkeypatch.setenv("LEO2D_SELL_TMAX", tmax)
    monkeypatch.setenv("LEO2D_SELL_UCAP", ucap)
    dev = L.Device(0)
    geom = L.Geometry(L.Deck(text))
    dev.set_geometry(geom)
    dev.pairs_build()
    dev.assemble(geom.jobs()[0], L.PATTERN_PRUNED)
    print("case", name, ucap, geom.n, flush=True)
    rp, ci, v = dev.csr_copy()
    M, R = 24, 32
    omu = oracle_mod.kpm(rp, ci, v, M, vecs=oracle_mod.random_phase(geom.n, R, 9), doubling_all=True, nthreads=8)
    for prec, tol in ((L.PREC_FP64, 1e-12), (L.PREC_MIXED, 2e-5)):
        mu = dev.kpm(M, random_phase=(R, 9), scheme=L.SCHEME_DOUBLING, precision=prec)
        assert dev.timing().kernel == 21, "a tile layout"
        assert np.max(np.abs(mu - omu)) <= tol * geom.n, prec


@pytest.mark.parametrize("pattern", [L.PATTERN_REFERENCE, L.PATTERN_PRUNED])
def test_long_rows_run_the_csr_step(oracle_mod, monkeypatch, pattern):
    monkeypatch.setenv("LEO2D_KPM_VARIANT", "20")
    dev = L.Device(0)
    geom = L.Geometry(L.Deck(W.tblg_flake_deck(5.0, 24.0, M=16)))
    dev.set_geometry(geom)
    dev.pairs_build()
    dev.assemble(geom.jobs()[0], pattern)
    rp, ci, v = dev.csr_copy()
    fits = int(np.max(np.diff(rp))) <= 64
    print("case", pattern, geom.n, "longest row", int(np.max(np.diff(rp))), flush=True)
    M, R = 24, 32
    omu = oracle_mod.kpm(rp, ci, v, M, vecs=oracle_mod.random_phase(geom.n, R, 9), doubling_all=True, nthreads=8)
    for _ in range(2):   # built (or refused) once, then kept
        mu = dev.kpm(M, random_phase=(R, 9), scheme=L.SCHEME_DOUBLING)
        assert dev.timing().kernel == (21 if fits else 14)
        assert np.max(np.abs(mu - omu)) <= 1e-12 * geom.n


@pytest.mark.parametrize("tiles", [1, 2, 3])
@pytest.mark.parametrize("R", [16, 32, 64])
@pytest.mark.parametrize("bloch", [0, 1])
def test_default_step_by_rows(oracle_mod, monkeypatch, tiles, R, bloch):
    """508, 2,032 and 4,572 rows: on either side of the least rows of the tiled
    step, each default against the oracle, and the FP32 recursion against the
    wavefront-per-row (or lane-per-vector) step, which sums rows alike."""
    monkeypatch.delenv("LEO2D_KPM_VARIANT", raising=False)
    dev = L.Device(0)
    geom = L.Geometry(L.Deck(W.tblg_cell_deck(7, 6, tiles)))
    dev.set_geometry(geom)
    dev.pairs_build()
    job = geom.jobs()[0]
    job.energy_rescale = 10.5   # the smallest cell's spectrum is the widest
    job.complex_matrix = bloch
    if bloch:
        job.k[0], job.k[1] = 0.011, -0.004
    dev.assemble(job, L.PATTERN_PRUNED)
    print("case", geom.n, R, bloch, flush=True)
    rp, ci, v = dev.csr_copy()
    M = 24
    omu = oracle_mod.kpm(rp, ci, v, M, vecs=oracle_mod.random_phase(geom.n, R, 9), doubling_all=True, nthreads=8)
    tiled = geom.n >= (2048 if R == 64 else 4096)
    mu = dev.kpm(M, random_phase=(R, 9), scheme=L.SCHEME_DOUBLING)
    assert dev.timing().kernel == (21 if tiled else 14)
    assert np.max(np.abs(mu - omu)) <= 1e-12 * geom.n
    mu32 = dev.kpm(M, random_phase=(R, 9), scheme=L.SCHEME_DOUBLING, precision=L.PREC_MIXED)
    monkeypatch.setenv("LEO2D_KPM_VARIANT", "1" if R == 64 else "0")
    ref32 = dev.kpm(M, random_phase=(R, 9), scheme=L.SCHEME_DOUBLING, precision=L.PREC_MIXED)
    assert np.max(np.abs(mu32 - ref32)) <= 1e-12 * geom.n
