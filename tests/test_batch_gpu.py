"""Batched 2D modelling of shots with uneven grids and lengths: every shot bit-exact against the
oracle's afd2d, with and without hipGraph capture; graph replays (with eager work and
synchronisations between them) reproduce the eager result exactly."""
import numpy as np
import pytest

import pywave_amd
from oracle import oracle as O
from pywave_amd import Afd2dBatch

pytestmark = pytest.mark.gpu


def _shots(seed, n):
    rng = np.random.default_rng(seed)
    shots = []
    for _ in range(n):
        nz, nx = int(rng.integers(18, 70)), int(rng.integers(20, 90))
        nt = int(rng.integers(60, 200))
        vel = (1500 + 2500 * rng.random((nz, nx))).astype(np.float32)
        ns = int(rng.integers(1, 3))
        sx = rng.integers(0, nx, ns).astype(np.float32)
        sz = rng.integers(0, nz, ns).astype(np.float32)
        f = rng.uniform(15, 35, ns).astype(np.float32)
        t = rng.uniform(0.0, 0.04, ns).astype(np.float32)
        A = rng.uniform(-1, 1, ns).astype(np.float32)
        wav = O.ricker_bank(nt, 0.001, f, t, A)
        shots.append(dict(vel=vel, d=(10.0, 12.0), nt=nt, dt=0.001, ns=ns,
                          src=np.concatenate([sx, sz, f, t, A]).astype(np.float32), wavelet=wav))
    return shots


def _oracle(s, nbt, ct):
    ns = s["ns"]
    src = s["src"]
    d, _, _ = O.afd2d(s["vel"], s["nt"], s["dt"], s["d"][1], s["d"][0], nbt, ct, src[:ns], src[ns:2 * ns],
                      s["wavelet"])
    return d.T  # (nt, nx)


@pytest.mark.parametrize("use_graph", [False, True])
def test_batch_shots_bit_exact(use_graph):
    shots = _shots(1, 7)
    b = Afd2dBatch(shots, nbt=6, ct=0.03)
    b.run(use_graph)
    for i, s in enumerate(shots):
        assert np.array_equal(b.traces(i), _oracle(s, 6, 0.03)), i


def test_graph_replays_match_eager():
    shots = _shots(2, 5)
    b = Afd2dBatch(shots, nbt=5, ct=0.02)
    b.run(False)
    ref = [b.traces(i) for i in range(len(shots))]
    for _ in range(3):
        b.run(True)
        # eager work between replays
        b2 = Afd2dBatch(shots[:2], nbt=5, ct=0.02)
        b2.run(False)
        b2.close()
        for i in range(len(shots)):
            assert np.array_equal(b.traces(i), ref[i])


def test_batch_matches_dropin_with_builtin_wavelet():
    rng = np.random.default_rng(4)
    shots = []
    for k in range(3):
        nz, nx, nt = 40 + 7 * k, 50 + 11 * k, 150 + 20 * k
        vel = (1800 + 900 * rng.random((nz, nx))).astype(np.float32)
        shots.append(dict(vel=vel, d=(10.0, 10.0), nt=nt, dt=0.001, ns=1,
                          src=np.array([nx // 2, 3, 20.0, 0.03, 1.0], np.float32)))
    out = pywave_amd.afd2d_batch(shots, nbt=10, ct=0.02)
    for s, tr in zip(shots, out):
        nz, nx = s["vel"].shape
        ref = pywave_amd.afd2d(s["vel"], nt=s["nt"], dt=0.001, ax=[0, 10, nx], az=[0, 10, nz], ns=1,
                               sx=[nx // 2], sz=[3], f=[20], t=[0.03], A=[1], nbt=10, ct=0.02, jsnap=0)
        assert np.array_equal(tr, ref.reshape(s["nt"], nx, order="F"))


def test_every_tile_width_bit_exact_and_tuning_recorded():
    # shots wide enough that every width has lean interior tiles beside general ones
    shots = _shots(5, 4) + [dict(_shots(6, 1)[0], vel=np.full((40, 150), 2500, np.float32))]
    ref = [_oracle(s, 6, 0.03) for s in shots]
    b = Afd2dBatch(shots, nbt=6, ct=0.03)
    b.run(True)
    w, log = b.width()
    assert w in (2, 4, 8, 16) and sorted(x for x, _ in log) == [2, 4, 8, 16] and all(ms > 0 for _, ms in log)
    for i in range(len(shots)):
        assert np.array_equal(b.traces(i), ref[i]), ("tuned", w, i)
    for xc in (2, 4, 8, 16):
        b.set_width(xc)
        b.run(True)
        assert b.width()[0] == xc
        for i in range(len(shots)):
            assert np.array_equal(b.traces(i), ref[i]), (xc, i)
    with pytest.raises(ValueError):
        b.set_width(3)
    b.close()
    # a second batch of the same geometry on the context takes the first one's choice and log
    b2 = Afd2dBatch(shots, nbt=6, ct=0.03)
    b2.run(False)
    assert b2.width() == (w, log)
    b2.close()


@pytest.mark.parametrize("nx,nt", [(128, 256), (33, 993), (181, 182), (1, 33000)])
def test_traces_transposed_on_host_and_device_vs_single_plans(nx, nt):
    # 32768 samples (the most that the host transposes), one more, and sizes off the 32 x 32 tiles of the
    # device's transpose: the single plans' traces, in the same order
    rng = np.random.default_rng(nx)
    vel = (1500 + 1500 * rng.random((12, nx))).astype(np.float32)
    src = np.array([nx // 2, 5, 20, 0.002, 1], np.float32)
    wav = rng.standard_normal((1, nt)).astype(np.float32)
    b = pywave_amd.Afd2dBatch([dict(vel=vel, d=(10.0, 10.0), nt=nt, dt=0.001, src=src, ns=1, wavelet=wav)], nbt=5)
    b.run()
    p = pywave_amd.AfdPlan(vel, (10.0, 10.0), nt, 0.001, 5, 0.01, 0)
    p.set_sources(src, 1, wavelet=wav)
    p.run()
    assert np.array_equal(b.traces(0), p.output().reshape(nt, nx, order="F"))
    b.close()
    p.close()
