"""Captured batched recursions whose row tiles are laid out again between two
replays: a replay reads the tiles of its own call, bit for bit as eager launches."""
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
