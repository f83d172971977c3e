"""Conductivity moments of blocks of up to four targets, whose two recursions run
in one launch, against the wider blocks that run them apart: the sums of a row go
in the same order, so each target's moments agree to rounding of the GEMM's chunk
sums (1e-12 of the largest), whatever block it sits in."""
import numpy as np
import pytest

import leo2d_amd as L
from leo2d_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("radius", [4.0, 13.0, 40.0])
@pytest.mark.parametrize("M", [2, 3, 24])
def test_pair_matches_separate(radius, M):
    dev = L.Device(0)
    geom = L.Geometry(L.Deck(W.tblg_flake_deck(3.0, radius, M=64)))
    dev.set_geometry(geom)
    dev.assemble_velocity(geom.jobs()[0], L.PATTERN_PRUNED)
    targets = [int(t) for t in np.linspace(0, geom.n - 1, 7)]
    print("case", geom.n, M, flush=True)
    ref = dev.cond_moments(M, targets, block=8)
    for block in (1, 2, 4):
        got = dev.cond_moments(M, targets, block=block)
        assert np.max(np.abs(got - ref)) <= 1e-12 * np.max(np.abs(ref)), block
    dev.close()


@pytest.mark.parametrize("radius", [13.0, 60.0])
def test_sixteen_targets(radius):
    """Blocks of 16 on fewer and on more rows than their launch covers in one round."""
    dev = L.Device(0)
    geom = L.Geometry(L.Deck(W.tblg_flake_deck(3.0, radius, M=64)))
    dev.set_geometry(geom)
    dev.assemble_velocity(geom.jobs()[0], L.PATTERN_PRUNED)
    targets = [int(t) for t in np.linspace(0, geom.n - 1, 17)]
    print("case", geom.n, flush=True)
    ref = dev.cond_moments(12, targets, block=4)
    got = dev.cond_moments(12, targets, block=16)
    assert np.max(np.abs(got - ref)) <= 1e-12 * np.max(np.abs(ref))
    dev.close()
