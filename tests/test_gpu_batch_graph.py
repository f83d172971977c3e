"""Captured batched recursions whose row tiles are laid out again between two
replays, and recursions that reduce their partials several times on the way: bit
for bit the eager launches and the run with one reduction."""
import numpy as np
import pytest

import leo2d_amd as L
from leo2d_amd import workloads as W

pytestmark = pytest.mark.gpu

M, R, SEED = 32, 16, 5


def _stack(dev, cells):
    for i in cells:
        geom = L.Geometry(L.Deck(W.tblg_cell_deck(i + 1, i, M=M)))
        dev.set_geometry(geom)
        dev.pairs_build()
        W.assemble_rescaled(dev, geom, (0.31, 0.12))
        dev.batch_append()


@pytest.mark.parametrize("first", ["1", "0"])
def test_replay_after_tiles_are_laid_out_again(monkeypatch, first):
    """The copy-wavefront form and the other take tiles of different heights, so a call
    of one between two of the other builds the stack's tiles twice in between."""
    other = "0" if first == "1" else "1"
    dev = L.Device(0)
    _stack(dev, (3, 5, 9))
    call = dict(seed=SEED, mode=L.BATCH_SELL)
    eager = {}
    for cw in (first, other):
        monkeypatch.setenv("LEO2D_SELL_CW", cw)
        eager[cw] = dev.batch_kpm(M, R, graph=False, **call)
    for rep in range(3):
        monkeypatch.setenv("LEO2D_SELL_CW", first)
        for _ in range(2):
            assert np.array_equal(dev.batch_kpm(M, R, graph=True, **call), eager[first]), rep
        monkeypatch.setenv("LEO2D_SELL_CW", other)
        assert np.array_equal(dev.batch_kpm(M, R, graph=False, **call), eager[other]), rep
        dev.kpm(16, random_phase=(8, rep), scheme=L.SCHEME_DOUBLING)   # takes and returns kept buffers
    dev.close()


@pytest.mark.parametrize("mode,Rv", [(L.BATCH_ROW_GROUPS, 4), (L.BATCH_ROW_GROUPS, 16), (L.BATCH_ENTRY_SLOTS, 16),
                                     (L.BATCH_ROW_CHUNKS, 16), (L.BATCH_SELL, 16), (L.BATCH_SELL, 32)])
@pytest.mark.parametrize("graph", [False, True])
def test_reductions_on_the_way(monkeypatch, mode, Rv, graph):
    """Cells of 76, 148 and 364 orbitals are 38 tiles of 16 rows, the most a call may cut:
    room for the partials of 1, 2 and 7 steps of them (some more of the higher SELL tiles),
    then for all 32."""
    dev = L.Device(0)
    _stack(dev, (2, 3, 5))
    kw = dict(seed=SEED, mode=mode, graph=graph)
    if mode != L.BATCH_SELL:
        kw["tile_rows"] = 16
    monkeypatch.delenv("LEO2D_PARTIAL_SPACE", raising=False)
    ref = dev.batch_kpm(64, Rv, **kw)
    for steps in (1, 2, 7):
        monkeypatch.setenv("LEO2D_PARTIAL_SPACE", str(steps * 38 * Rv * 16))
        for _ in range(3 if graph else 1):
            assert np.array_equal(dev.batch_kpm(64, Rv, **kw), ref), steps
            dev.kpm(16, random_phase=(4, steps), scheme=L.SCHEME_DOUBLING)
    dev.close()


@pytest.mark.parametrize("R,kernel", [(4, 2), (16, 14), (32, 21), (64, 1)])
def test_single_recursion_reductions_on_the_way(monkeypatch, R, kernel):
    """The same for one Hamiltonian on eight workgroups: 192 bytes a step and vector."""
    monkeypatch.setenv("LEO2D_KPM_VARIANT", {21: "20"}.get(kernel, str(kernel)))
    dev = L.Device(0)
    geom = L.Geometry(L.Deck(W.tblg_cell_deck(6, 5, M=64)))
    dev.set_geometry(geom)
    W.assemble_rescaled(dev, geom, (0.31, 0.12))
    t = np.arange(R, dtype=np.int32) * 5
    for kw in (dict(targets=t), dict(random_phase=(R, 3)), dict(random_phase=(R, 3), scheme=L.SCHEME_DOUBLING)):
        monkeypatch.delenv("LEO2D_PARTIAL_SPACE", raising=False)
        ref = dev.kpm(64, grid=8, **kw)
        assert dev.timing().kernel == kernel
        for steps in (1, 2, 7):
            monkeypatch.setenv("LEO2D_PARTIAL_SPACE", str(steps * R * 192))
            assert np.array_equal(dev.kpm(64, grid=8, **kw), ref), steps
    dev.close()
