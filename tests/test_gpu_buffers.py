"""Device buffers a handle keeps between calls: calls of other sizes and kinds in
between, and other handles on other threads, leave every result bit for bit what
a fresh handle gives."""
import ctypes as C
import threading

import numpy as np
import pytest

import leo2d_amd as L
from leo2d_amd import workloads as W

pytestmark = pytest.mark.gpu


def _calls(dev):
    """Moments and DoS of matrices of several sizes, conductivity and a batch, in one sequence."""
    out = []
    for radius, R in ((12.0, 3), (30.0, 16), (12.0, 1), (21.0, 64), (12.0, 3)):
        geom = L.Geometry(L.Deck(W.tblg_flake_deck(3.0, radius, M=64)))
        dev.set_geometry(geom)
        job = geom.jobs()[0]
        dev.assemble_velocity(job, L.PATTERN_PRUNED)
        mu = dev.kpm(64, targets=np.arange(R, dtype=np.int32))
        out += [mu, dev.dos(mu, 10.5, 0.0)[1], dev.kpm(64, random_phase=(R, 5)), dev.cond_moments(24, [0, 1, 2])]
        dev.batch_append()
    out.append(dev.batch_kpm(32, 16, seed=3, mode=L.BATCH_ROW_CHUNKS))
    dev.batch_clear()
    return out


def _fresh():
    dev = L.Device(0)
    try:
        return _calls(dev)
    finally:
        dev.close()


def test_repeated_calls_on_kept_buffers():
    ref = _fresh()
    dev = L.Device(0)
    for _ in range(3):
        assert all(np.array_equal(a, b) for a, b in zip(_calls(dev), ref))
    dev.close()


def test_handles_on_threads():
    ref = _fresh()
    got = [None] * 3

    def work(k):
        got[k] = [_fresh(), _fresh()]

    threads = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for pair in got:
        for calls in pair:
            assert all(np.array_equal(a, b) for a, b in zip(calls, ref))


def test_ensemble_members_destroyed_in_any_order():
    x = np.random.default_rng(0).standard_normal((700, 72)).astype(np.float32)
    nets = [L.Mlp(0, 72, 64, 2, 96, seed=k) for k in range(3)]
    one = [m.forward(x) for m in nets]
    mean, spread = L.mlp_ensemble([nets[1], nets[0], nets[2], nets[0]], x)
    ref = np.mean([one[1], one[0], one[2], one[0]], axis=0)
    assert np.max(np.abs(mean - ref)) <= 1e-6 * np.max(np.abs(ref))
    nets[1].close()
    assert np.array_equal(nets[0].forward(x), one[0])
    nets[0].close()
    assert np.array_equal(nets[2].forward(x), one[2])
    nets[2].close()


def test_large_buffers_of_many_handles():
    """Six handles with vector sets of 0.8 GB each pass the 4 GiB the process keeps: the
    later ones' sets are freed, or push out what their own handle kept."""
    geom = L.Geometry(L.Deck(W.tblg_flake_deck(1.05, 100.0, M=64)))
    devs, ref = [], None
    for _ in range(6):
        dev = L.Device(0)
        devs.append(dev)
        dev.set_geometry(geom)
        dev.assemble_velocity(geom.jobs()[0], L.PATTERN_PRUNED)
        for M in (512, 384, 512):
            got = dev.cond_moments(M, [0, 100, 1000, 10000])
        ref = got if ref is None else ref
        assert np.array_equal(got, ref)
    for dev in devs:
        dev.close()


def _free_bytes():
    free, total = C.c_size_t(), C.c_size_t()
    assert L.lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0   # the runtime the library runs on
    return free.value


def test_batch_clear_gives_memory_back():
    """A stack of 571,584 rows with blocks of 32 vectors takes some 1.2 GB; after the clear
    the device has all but 256 MiB of it again."""
    dev = L.Device(0)
    geom = L.Geometry(L.Deck(W.tblg_cell_deck(32, 31, 4, M=8)))
    dev.set_geometry(geom)
    W.assemble_rescaled(dev, geom, (0.2, 0.1))
    dev.batch_clear()
    before = _free_bytes()
    for _ in range(3):
        dev.batch_append()
    mu = dev.batch_kpm(8, 32, seed=1)
    during = _free_bytes()
    assert before - during > 900 << 20
    dev.batch_clear()
    after = _free_bytes()
    assert before - after <= 320 << 20   # and what the runtime rounds up
    for _ in range(3):
        dev.batch_append()
    assert np.array_equal(dev.batch_kpm(8, 32, seed=1), mu)
    dev.close()
