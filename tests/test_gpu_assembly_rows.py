"""The wavefront-per-row fill at row shapes where its 64-lane walk can go wrong:
runs of equal columns longer than a chunk's remainder (the smallest periodic
cells, every image of an orbital in one slot), rows whose supported slots are
fewer than 64, between 64 and 128 and more, and flakes of a few orbitals.
Pattern bit-exact; values within 1e-12 relative (the GPU's exp, sincos and
atan2 differ from glibc's by a few ulp), as in test_gpu_parity.py."""
import numpy as np
import pytest

import leo2d_amd as L
from leo2d_amd import workloads as W

pytestmark = pytest.mark.gpu

DECKS = {
    "cell_2_1": W.tblg_cell_deck(2, 1, M=16),
    "cell_2_1_graphene": W.tblg_cell_deck(2, 1, M=16).replace("GrapheneSimple", "Graphene"),
    "cell_3_2_graphene": W.tblg_cell_deck(3, 2, M=16).replace("GrapheneSimple", "Graphene"),
    "flake_3": W.tblg_flake_deck(5.0, 3, M=16),
    "flake_9_graphene": W.tblg_flake_deck(5.0, 9, M=16, material="Graphene"),
    "flake_18_graphene": W.tblg_flake_deck(5.0, 18, M=16, material="Graphene"),
}


@pytest.mark.parametrize("name", sorted(DECKS))
@pytest.mark.parametrize("pattern", [L.PATTERN_REFERENCE, L.PATTERN_PRUNED])
@pytest.mark.parametrize("bloch", [False, True])
def test_fill_rows(oracle_mod, name, pattern, bloch):
    text = DECKS[name]
    print("case", name, pattern, bloch, flush=True)
    dev = L.Device(0)
    geom = L.Geometry(L.Deck(text))
    dev.set_geometry(geom)
    dev.pairs_build()
    job = geom.jobs()[0]
    od = oracle_mod.parse_deck(text)
    oracle_mod.setup_supercell(od)
    og = oracle_mod.Geometry(oracle_mod.geom_desc(od))
    oj = oracle_mod.make_job(od, oracle_mod.build_jobs(od, oracle_mod.target_list(od, og))[0], pruned=pattern)
    if bloch:
        for j in (job, oj):
            j.complex_matrix = 1
            j.k[0], j.k[1] = 0.31, -0.17
    dev.assemble_velocity(job, pattern)
    rp, ci, v = dev.csr_copy()
    dx, dy = dev.velocity_copy(with_dy=True)
    orp, oci, ov, odx, ody = og.assemble(oj, with_dx=True, with_dy=True)
    assert np.array_equal(rp, orp) and np.array_equal(ci, oci)
    for a, b in ((v, ov), (dx, odx), (dy, ody)):
        assert np.all(np.abs(a - b) <= 1e-12 * np.abs(b) + 1e-13 * np.max(np.abs(b)))
    dev.close()
