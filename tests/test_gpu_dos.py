"""The DoS transform's direct sum on the GPU against the oracle: lengths at the
edges of its wavefront slices, column blocks and LDS table, and row counts at
the edges of a row group."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    import leo2d_amd as L

    d = L.Device(0)
    yield d
    d.close()


@pytest.mark.parametrize("T,M", [(1, 2), (3, 3), (8, 15), (9, 16), (1, 127), (2, 128), (7, 130), (17, 500), (4, 2049),
                                 (2, 8192), (1, 20004)])
def test_dos_lengths_and_rows(dev, T, M):
    """Every term is at most |g mu| and carries a phase exact to one rounding, so a
    row's sum is good to about M rounding units of its largest term: 1e-15 M of
    the largest moment, with the density's prefactor on top."""
    from oracle import oracle as orc

    rng = np.random.default_rng(M)
    mu = rng.standard_normal((T, M)) / (1.0 + np.arange(M))
    E, rho = dev.dos(mu, 7.5, 0.25, scale=0.5)
    ref = 0.5 * orc.dos(mu, 7.5, 0.25)
    k = np.arange(M)
    assert np.max(np.abs(E - (0.25 + 7.5 * np.cos((k + 0.5) * np.pi / M)))) <= 1e-14 * 8
    pre = 0.5 / (np.pi * np.sqrt(7.5 ** 2 - (E - 0.25) ** 2))
    assert np.all(np.abs(rho - ref) <= 4e-15 * max(M, 64) * np.max(np.abs(mu)) * pre + 1e-9 * np.abs(ref))
