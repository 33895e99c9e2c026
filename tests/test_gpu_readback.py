"""Results on their way to the host: transposed and packed on the device, the model gradients combined
there (csrc/readback.hip).

Traces and wavefields are moved, so they are bit-equal to another way of getting the same values. The
model gradients are FP64 sums of at most 30 products of the coefficient gradients with factors of at
most 12 roundings each; against the same sums in numpy both sides differ by at most
2 * (30 + 12) * 2^-53 of the sum of the terms' magnitudes.
"""
import numpy as np
import pytest

import wavesim
from wavesim import cases

pytestmark = pytest.mark.gpu

CHAIN_TOL = 2 * (30 + 12) * 2.0 ** -53


def _shot(rng, n, NT, nrec, nsrc=1, ntype=3):
    sig = rng.standard_normal((nsrc, NT)).astype(np.float32)
    s = cases.Shot(rng.integers(0, n, nsrc), rng.integers(1, ntype + 1, nsrc).astype(np.int32), sig,
                   rng.integers(0, n, nrec), rng.integers(1, ntype + 1, nrec).astype(np.int32))
    s.rec_index[:nsrc], s.rec_type[:nsrc] = s.src_index[:nrec], s.src_type[:nrec]
    return s


def _solver(dim, type_, shape, NT, shots, m=(2000.0, 1100.0, 2100.0), order=4, **settings):
    NX, NY, NZ = shape
    n = NX * NY * NZ
    fs = wavesim.create(dim, type_)
    fs.init_forward_solver(NX=NX, NY=NY, NZ=NZ, NT=NT, DH=1.0, DT=1e-4, spatial_fd_order=order, nshots=len(shots),
                           **settings)
    m = [np.broadcast_to(np.asarray(k, np.float32), (n,)) for k in m]
    fs.prepare_for_modelling(m[0], None if type_ == "acoustic" else m[1], m[2])
    for k, s in enumerate(shots):
        fs.set_acquisition(k, s.src_index, s.src_type, s.src_signal, s.rec_index, s.rec_type)
    return fs


@pytest.mark.parametrize("dim,shape", [("2D", (71, 50, 1)), ("3D", (19, 14, 17))])
@pytest.mark.parametrize("NT", [1, 64, 129])
def test_traces_of_uneven_shots(dim, shape, NT):
    """Tile edges in time and traces, a shot without receivers: each trace equals the same receiver's in
    a handle that holds this shot alone with its receivers in reverse order."""
    rng = np.random.default_rng(NT)
    n = int(np.prod(shape))
    shots = [_shot(rng, n, NT, k, nsrc=5) for k in (1, 63, 0, 64, 193)]
    fs = _solver(dim, "acoustic", shape, NT, shots)
    fs.run(0, NT)
    got = [fs.seismograms(k) for k in range(len(shots))]
    for k, s in enumerate(shots):
        assert got[k].shape == (len(s.rec_index), NT)
        one = cases.Shot(s.src_index, s.src_type, s.src_signal, s.rec_index[::-1], s.rec_type[::-1])
        ref = _solver(dim, "acoustic", shape, NT, [one])
        ref.run(0, NT)
        assert np.array_equal(got[k], ref.seismograms(0)[::-1])
        assert np.array_equal(fs.seismograms(k), got[k])
    assert max(np.abs(g).max() for g in got if g.size) > 0


def test_traces_in_parts():
    """More than the staging buffer's 64 MiB: 17,000 traces of 1000 steps; repeated receivers agree."""
    rng = np.random.default_rng(3)
    NT, n = 1000, 40 * 30
    s = _shot(rng, n, NT, 1700)
    s.rec_index, s.rec_type = np.tile(s.rec_index, 10), np.tile(s.rec_type, 10)
    fs = _solver("2D", "acoustic", (40, 30, 1), NT, [s])
    fs.run(0, NT)
    d = fs.seismograms(0).reshape(10, 1700, NT)
    assert np.abs(d[0]).max() > 0
    assert all(np.array_equal(d[0], d[k]) for k in range(1, 10))


@pytest.mark.parametrize("dim,type_,shape", [("2D", "elastic", (8, 8, 1)), ("2D", "acoustic", (65, 3, 1)),
                                             ("2D", "sh", (127, 41, 1)), ("2D", "elastic", (4200, 4100, 1)),
                                             ("3D", "acoustic", (33, 20, 18)), ("3D", "elastic", (18, 21, 16))])
def test_wavefield_round_trip(dim, type_, shape):
    rng = np.random.default_rng(5)
    n = int(np.prod(shape))
    if type_ == "sh":
        fs = wavesim.create(dim, type_)
        fs.init_forward_solver(NX=shape[0], NY=shape[1], NT=4, DH=1.0, DT=1e-4, spatial_fd_order=4, nshots=2)
        fs.prepare_for_modelling(None, np.full(n, 900.0, np.float32), np.full(n, 2000.0, np.float32))
    else:
        fs = _solver(dim, type_, shape, 4, [_shot(rng, n, 4, 0)] * 2)
    v = [rng.standard_normal(n).astype(np.float32) for _ in range(2)]
    for k in range(2):
        fs.set_wavefield(0, v[k], k)
    for k in range(2):
        assert np.array_equal(fs.wavefield(0, k).reshape(-1), v[k])


def _chain(dim, param, shape, c, vp, vs, rho, magnitude):
    """Scatter form of the chain rule: coefficient gradients c (each [NY][NZ][NX]) -> vp, vs or rho."""
    axis = {0: 2, 1: 0, 2: 1}  # model direction x, y, z -> array axis
    vp, vs, rho = (a.astype(np.float64).reshape(c[0].shape) for a in (vp, vs, rho))
    sgn = 1.0 if magnitude else -1.0
    raw = rho * vs * vs
    mu = np.maximum(raw, 1.0)

    def sl(ax, lo, hi):
        s = [slice(None)] * 3
        s[ax] = slice(lo, hi)
        return tuple(s)

    def plus(a, ax):  # value of the next cell along ax, 0 beyond the grid
        out = np.zeros_like(a)
        out[sl(ax, 0, -1)] = a[sl(ax, 1, None)]
        return out

    def back(a, ax):  # scatter to the next cell along ax
        out = np.zeros_like(a)
        out[sl(ax, 1, None)] = a[sl(ax, 0, -1)]
        return out

    if param == 0:
        return c[dim] * 2 * rho * vp
    gmu = c[dim + 1].copy()
    for pl, (a0, a1) in enumerate([(0, 1)] if dim == 2 else [(0, 1), (0, 2), (1, 2)]):
        a0, a1 = axis[a0], axis[a1]
        inv, one = 1.0 / mu, np.ones_like(mu)
        s = inv + plus(inv, a0) + plus(inv, a1) + plus(plus(inv, a0), a1)
        cnt = one + plus(one, a0) + plus(one, a1) + plus(plus(one, a0), a1)
        m = cnt / s
        t = np.where(m < 4.0, 0.0, c[dim + 2 + pl] * m * m / cnt)
        gmu += (t + back(t, a0) + back(t, a1) + back(back(t, a0), a1)) / (mu * mu)
    if param == 1:
        return np.where(raw >= 1.0, gmu * 2 * rho * vs, 0.0)
    g = c[dim] * vp * vp + np.where(raw >= 1.0, gmu * vs * vs, 0.0)
    for k in range(dim):
        ax = axis[k]
        av = 0.5 * (rho + plus(rho, ax))
        t = sgn * c[k] * 0.5 / (av * av)
        t[sl(ax, -1, None)] = 0.0
        g += t + back(t, ax)
        g[sl(ax, -1, None)] += sgn * c[k][sl(ax, -1, None)] / rho[sl(ax, -1, None)] ** 2
    return g


@pytest.mark.parametrize("dim,shape", [("2D", (67, 53, 1)), ("2D", (9, 8, 1)), ("2D", (2900, 3000, 1)),
                                       ("3D", (19, 17, 18))])
def test_model_gradient_is_the_chain_rule(dim, shape):
    """Also beyond the staging buffer's size (rows that two parts share), at the last cells, and where
    the shear modulus is clamped or its average set to zero."""
    rng = np.random.default_rng(11)
    NX, NY, NZ = shape
    n, d = NX * NY * NZ, int(dim[0])
    NT = 12 if n > 1 << 20 else 40
    vp = (2000.0 * (1 + 0.1 * rng.random(n))).astype(np.float32)
    vs = (1100.0 * (1 + 0.1 * rng.random(n))).astype(np.float32)
    rho = (2100.0 * (1 + 0.1 * rng.random(n))).astype(np.float32)
    x = np.arange(n) % NX
    vs[(x >= NX // 2) & (x < NX // 2 + 4)] = 0.0
    vs[x == NX // 2 + 1] = 0.01   # mu clamped to 1
    vs[x == NX // 2 + 2] = 0.03   # above the clamp, averages below 4
    rows = np.arange(0, NY, 2)
    cells = rows * NX * NZ + rows % NZ * NX + (rows * 3) % NX
    typ = (np.arange(len(cells)) % (d + 1) + 1).astype(np.int32)
    sig = rng.standard_normal((len(cells), NT)).astype(np.float32)
    fs = wavesim.create(dim, "elastic")
    fs.init_forward_solver(NX=NX, NY=NY, NZ=NZ, NT=NT, DH=1.0, DT=1e-4, spatial_fd_order=2, nshots=1)
    fs.prepare_for_modelling(vp, vs, rho)
    fs.set_acquisition(0, cells, typ, sig, cells, typ)
    fs.set_checkpointing(every=10, fp16=False)
    fs.run(0, NT)
    fs.set_adjoint_source(0, fs.seismograms(0))
    fs.run_adjoint()
    nc = 5 if d == 2 else 8
    c = [np.asarray(fs.gradient(3 + k)).reshape(NY, NZ, NX) for k in range(nc)]
    assert all(np.abs(k).max() > 0 for k in c)
    for param, name in enumerate(("vp", "vs", "rho")):
        want = _chain(d, param, shape, c, vp, vs, rho, False)
        size = _chain(d, param, shape, [np.abs(k) for k in c], vp, vs, rho, True)
        got = np.asarray(fs.gradient(name)).reshape(NY, NZ, NX)
        assert np.abs(got).max() > 0
        assert np.all(np.abs(got - want) <= CHAIN_TOL * size), name
