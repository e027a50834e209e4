"""HIP pseudo-spectral engine (aps2d/aps3d) against the compiled reference's golden vectors and the
oracle.

Bar: bit-exact (np.array_equal, +0 == -0): the device transforms reproduce the reference's KISS FFT
arithmetic, so traces, snapshots and time-reversal fields equal the reference's, through the
resident plan fed the reference's wavelet and through the drop-in aps2d/aps3d."""
import numpy as np
import pytest

import pywave_amd
from oracle import oracle as O
from pywave_amd import AfdPlan
from pywave_amd import _native as N

pytestmark = pytest.mark.gpu


def _plan(g, ndim):
    d = (float(g["dz"]), float(g["dx"])) + ((float(g["dy"]),) if ndim == 3 else ())
    return AfdPlan(g["vel"], d, int(g["nt"]), float(g["dt"]), int(g["nbt"]), float(g["ct"]), int(g["jsnap"]),
                   spectral=True)


def test_aps2d_golden_bit_exact(golden):
    g = golden("aps2d_two_sources")
    p = _plan(g, 2)
    p.set_sources(g["src"], len(g["src"]) // 5, wavelet=g["rick"])
    p.run()
    assert np.array_equal(p.output(), g["out"])
    # the drop-in, with its own wavelet
    src = g["src"]
    ns = len(src) // 5
    nz, nx = g["vel"].shape
    dout, wfd = pywave_amd.aps2d(g["vel"], nt=int(g["nt"]), dt=float(g["dt"]), ax=[0, float(g["dx"]), nx],
                                 az=[0, float(g["dz"]), nz], ns=ns, sx=src[:ns], sz=src[ns:2 * ns],
                                 f=src[2 * ns:3 * ns], t=src[3 * ns:4 * ns], A=src[4 * ns:], nbt=int(g["nbt"]),
                                 ct=float(g["ct"]), jsnap=int(g["jsnap"]), verb=False)
    nt = int(g["nt"])
    assert np.array_equal(dout, g["out"][:nt * nx].reshape(nt, nx, order="F"))
    assert np.array_equal(wfd, g["out"][nt * nx:].reshape(nz, nx, -1, order="F"))


def test_aps2d_tri_golden_bit_exact(golden):
    g = golden("aps2d_tri")
    p = _plan(g, 2)
    p.set_tri_data(g["dat"])
    p.run(tri=True)
    assert np.array_equal(p.output(), g["out"])
    nz, nx = g["vel"].shape
    nt = int(g["nt"])
    w0 = g["out"][nt * nx:nt * nx + nz * nx].reshape(nz, nx, order="F")
    assert np.array_equal(p.final_field(), w0)


def test_aps3d_golden_bit_exact(golden):
    g = golden("aps3d_small")
    p = _plan(g, 3)
    p.set_sources(g["src"], len(g["src"]) // 6, wavelet=g["rick"])
    p.run()
    assert np.array_equal(p.output(), g["out"])
    src = g["src"]
    nz, nx, ny = g["vel"].shape
    nt = int(g["nt"])
    dout, wfd = pywave_amd.aps3d(g["vel"], nt=nt, dt=float(g["dt"]), ax=[0, float(g["dx"]), nx],
                                 ay=[0, float(g["dy"]), ny], az=[0, float(g["dz"]), nz], ns=1, sx=src[:1],
                                 sy=src[1:2], sz=src[2:3], f=src[3:4], t=src[4:5], A=src[5:6], nbt=int(g["nbt"]),
                                 ct=float(g["ct"]), jsnap=int(g["jsnap"]), verb=False)
    assert np.array_equal(dout, g["out"][:nt * nx * ny].reshape(nt, nx, ny, order="F"))


@pytest.mark.parametrize("shape,nbt", [((61, 83), 20), ((30, 44), 7), ((50, 31), 12)])
def test_aps2d_other_factorisations_vs_oracle(shape, nbt):
    # padded sizes 108x125 (2^2 3^3 x 5^3), 44x60, 80x60 ... exercise every butterfly radix on both
    # axes, against the oracle's transforms
    rng = np.random.default_rng(sum(shape))
    nz, nx = shape
    vel = (1500 + 1200 * rng.random(shape)).astype(np.float32)
    nt, dt, dx, dz = 180, 0.001, 10.0, 9.0
    sx, sz = [nx // 3, 2 * nx // 3], [nz // 2, nz // 4]
    rick = np.stack([O.ricker(nt, dt, 20, 0.03, 1.0), O.ricker(nt, dt, 15, 0.05, -0.7)]).astype(np.float32)
    d, snaps, _ = O.afd2d(vel, nt, dt, dx, dz, nbt, 0.02, sx, sz, rick, jsnap=45, ps=True)
    p = AfdPlan(vel, (dz, dx), nt, dt, nbt, 0.02, 45, spectral=True)
    pack = np.array(sx + sz + [20, 15] + [0.03, 0.05] + [1.0, -0.7], np.float32)
    p.set_sources(pack, 2, wavelet=rick)
    p.run()
    out = p.output()
    assert np.array_equal(out[:nt * nx].reshape(nt, nx, order="F"), d.T)
    w = out[nt * nx:].reshape(nz, nx, -1, order="F")
    assert all(np.array_equal(w[..., k], snaps[k].T) for k in range(w.shape[-1]))


def test_aps3d_other_factorisation_vs_oracle():
    rng = np.random.default_rng(21)
    nz, nx, ny = 17, 21, 25
    vel = (1700 + 900 * rng.random((nz, nx, ny))).astype(np.float32)
    nt, dt = 60, 0.001
    rick = O.ricker(nt, dt, 25, 0.02, 1.0)[None, :].astype(np.float32)
    d, _, _ = O.afd3d(vel, nt, dt, 10.0, 11.0, 12.0, 6, 0.03, [10], [12], [8], rick, ps=True)
    p = AfdPlan(vel, (12.0, 10.0, 11.0), nt, dt, 6, 0.03, 0, spectral=True)
    p.set_sources(np.array([10, 12, 8, 25, 0.02, 1.0], np.float32), 1, wavelet=rick)
    p.run()
    out = p.output()
    assert np.array_equal(out.reshape(nt, nx, ny, order="F"), d.transpose(2, 1, 0))


@pytest.mark.parametrize("shape", [(84, 83, 85), (147, 79, 90), (19, 115, 118), (3, 118, 115), (250, 3, 2)])
def test_aps3d_lines_per_block_vs_oracle(shape):
    # grids on which the z, x and y kernels run 16, 8, 4 and 1 lines per block (two levels a pass or
    # one), with partial last blocks and radix-5 lengths (125) on x or y; same operations in the same
    # order as the oracle, so equal
    rng = np.random.default_rng(sum(shape))
    nz, nx, ny = shape
    vel = (1700 + 900 * rng.random(shape)).astype(np.float32)
    nt, dt, nbt = 9, 0.001, 5
    wav = rng.standard_normal((1, nt)).astype(np.float32)
    s = [nx // 2, ny // 2, min(1, nz - 1)]
    d, snaps, _ = O.afd3d(vel, nt, dt, 10.0, 11.0, 12.0, nbt, 0.03, s[:1], s[1:2], s[2:], wav, jsnap=8, ps=True)
    p = AfdPlan(vel, (12.0, 10.0, 11.0), nt, dt, nbt, 0.03, 8, spectral=True)
    p.set_sources(np.array(s + [25, 0.002, 1.0], np.float32), 1, wavelet=wav)
    p.run()
    out = p.output()
    n = nt * nx * ny
    assert np.array_equal(out[:n].reshape(nt, nx, ny, order="F"), d.transpose(2, 1, 0))
    w = out[n:].reshape(nz, nx, ny, -1, order="F")
    assert all(np.array_equal(w[..., k], snaps[k].transpose(2, 1, 0)) for k in range(w.shape[-1]))


@pytest.mark.parametrize("shape,what", [((4000, 740, 740), "2^31 cells"), ((4700, 3, 3), "4680 samples"),
                                        ((8, 1830, 3), "1820 along x and y"), ((8, 3, 1830), "1820 along x and y")])
def test_spectral_extents_refused(shape, what):
    # padded grids of 2^31 cells or more (2.25e9 here) and lines beyond the kernels' lengths: refused
    # when the plan becomes spectral, before the operator is formed
    L, ctx = N.lib(), N.context()
    p = L.pw_afd_create(ctx, 3, *shape, 10.0, 10.0, 10.0, 1, 0.001, 0, 0.01, 0)
    assert p
    try:
        assert L.pw_afd_set_spectral(p, 1) == -1
        assert what in L.pw_last_error(ctx).decode()
    finally:
        L.pw_afd_destroy(p)


@pytest.mark.parametrize("shape", [(4490, 5), (2990, 7), (2420, 6), (2390, 6), (1300, 9), (6, 1790), (4490, 3, 4), (84, 85, 180)])
def test_aps_long_lines_vs_oracle(shape):
    # z columns of 512- and 256-thread blocks, up to 99 KB of LDS (2250 pairs; 66 KB at 1500) and more
    # cells than a block loads at once, an x line of 1800 points, and 190-point y lines whose operator
    # values take a second round of loads; same operations in the same order as the oracle's, so equal
    rng = np.random.default_rng(sum(shape))
    nt, dt, nbt, d2, d3 = 4, 0.0005, 5, (9.0, 10.0), (12.0, 10.0, 11.0)
    vel = (1700 + 900 * rng.random(shape)).astype(np.float32)
    wav = rng.standard_normal((1, nt)).astype(np.float32)
    s = [n // 2 for n in shape[1:]] + [min(1, shape[0] - 1)]
    if len(shape) == 2:
        d, snaps, _ = O.afd2d(vel, nt, dt, d2[1], d2[0], nbt, 0.03, s[:1], s[1:], wav, jsnap=3, ps=True)
    else:
        d, snaps, _ = O.afd3d(vel, nt, dt, d3[1], d3[2], d3[0], nbt, 0.03, s[:1], s[1:2], s[2:], wav, jsnap=3, ps=True)
    p = AfdPlan(vel, d2 if len(shape) == 2 else d3, nt, dt, nbt, 0.03, 3, spectral=True)
    p.set_sources(np.array(s + [25, 0.002, 1.0], np.float32), 1, wavelet=wav)
    p.run()
    out = p.output()
    n = nt * int(np.prod(shape[1:]))
    assert np.array_equal(out[:n].reshape((nt,) + shape[1:], order="F"), d.T)
    w = out[n:].reshape(shape + (-1,), order="F")
    assert all(np.array_equal(w[..., k], snaps[k].T) for k in range(w.shape[-1]))


@pytest.mark.parametrize("shape,ns", [((30, 25), 4), ((30, 25), 5), ((30, 25), 130), ((40, 6), 700), ((84, 83, 85), 300)])
def test_aps_many_sources_vs_oracle(shape, ns):
    # source counts on either side of those that a block of columns lists (more than 4 in all, up to 256
    # that reach it: 700 over six columns exceed that), several on one cell: added in source order as the
    # oracle does, so equal
    rng = np.random.default_rng(ns)
    nt, dt, nbt, d2, d3 = 5, 0.0005, 5, (9.0, 10.0), (12.0, 10.0, 11.0)
    vel = (1700 + 900 * rng.random(shape)).astype(np.float32)
    wav = rng.standard_normal((ns, nt)).astype(np.float32)
    s = [rng.integers(0, n, ns) for n in shape[1:] + shape[:1]]
    for c in s:
        c[-2:] = c[0]
    l = [list(c) for c in s]
    if len(shape) == 2:
        d, snaps, _ = O.afd2d(vel, nt, dt, d2[1], d2[0], nbt, 0.03, l[0], l[1], wav, jsnap=4, ps=True)
    else:
        d, snaps, _ = O.afd3d(vel, nt, dt, d3[1], d3[2], d3[0], nbt, 0.03, l[0], l[1], l[2], wav, jsnap=4, ps=True)
    p = AfdPlan(vel, d2 if len(shape) == 2 else d3, nt, dt, nbt, 0.03, 4, spectral=True)
    p.set_sources(np.concatenate(s + [np.full(ns, 25), np.full(ns, 0.002), np.ones(ns)]).astype(np.float32), ns, wavelet=wav)
    p.run()
    out = p.output()
    n = nt * int(np.prod(shape[1:]))
    assert np.array_equal(out[:n].reshape((nt,) + shape[1:], order="F"), d.T)
    w = out[n:].reshape(shape + (-1,), order="F")
    assert all(np.array_equal(w[..., k], snaps[k].T) for k in range(w.shape[-1]))
