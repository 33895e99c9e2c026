"""The resident 2D time loop (resident2d_kernel.hpp) against the two-launch kernels.

A handle that names no tile height may run its steps in the resident loop (fields in LDS, halos
exchanged between blocks); a handle with an explicit tile height runs the two-launch kernels, which
the other tests hold against the oracle.  Both do the same operations in the same order, so
seismograms and final wavefields are equal to the bit: at tile edges (columns 63 .. 129), few and
many rows, every order, CPML / ABS / rigid edges with and without a free surface, more sources than
a wavefront and more receivers than a block holds, several rounds of shots, runs cut into pieces,
queued runs, and the adjoint's record.
"""
import ctypes as C
import time

import numpy as np
import pytest

import wavesim
from wavesim import cases

pytestmark = pytest.mark.gpu

TWO = {"elastic": "strip", "acoustic": "phased", "sh": "phased", "tmem": "phased"}


def _case(physics, NX, NY, NT, order, nshots, damping, fs=0, W=8, ops=None):
    if physics == "elastic":
        c = cases.visco_2d(NX=NX, NY=NY, NT=NT, nshots=nshots, order=order, W=W, damping=damping, free_surface=fs)
        c.type, c.visco = "elastic", None
    elif physics == "sh":
        c = cases.sh_2d(NX=NX, NY=NY, NT=NT, nshots=nshots, order=order, W=W, damping=damping, free_surface=fs)
    elif physics == "tmem":
        c = cases.viscotmem_2d(NX=NX, NY=NY, NT=NT, nshots=nshots, order=order, W=W, damping=damping)
        c.type, c.visco = "tmem", None
    else:
        c = cases.visco_2d(NX=NX, NY=NY, NT=NT, nshots=nshots, order=order, W=W, damping=damping, free_surface=fs)
        c.type, c.visco, c.m1 = "acoustic", None, None
    return c


def _equal(c, NT, pieces=None, plan=None, **kw):
    a = cases.make_solver(c, **kw)
    if plan:
        assert a.resident_plan(*plan)[:2] == plan
    b = cases.make_solver(c, path=TWO[c.type], tile_y=16)
    cuts = [0] + (pieces or []) + [NT]
    for t0, t1 in zip(cuts[:-1], cuts[1:]):
        a.run(t0, t1)
    b.run(0, NT)
    for k in range(len(c.shots)):
        x, y = a.seismograms(k), b.seismograms(k)
        assert np.abs(y).max() > 0
        assert np.array_equal(x, y), (k, np.abs(x - y).max())
        for f in range(5 if c.type == "elastic" else 3):
            assert np.array_equal(a.wavefield(f, k), b.wavefield(f, k)), (k, f)


@pytest.mark.parametrize("physics", ["elastic", "acoustic", "sh", "tmem"])
@pytest.mark.parametrize("order,NX,NY,damping", [(2, 64, 40, 2), (4, 65, 33, 0), (6, 129, 97, 1), (8, 63, 150, 2),
                                                 (8, 190, 41, 1), (10, 128, 61, 2), (12, 131, 130, 2)])
def test_resident_equals_two_launch(physics, order, NX, NY, damping):
    _equal(_case(physics, NX, NY, 90, order, 2, damping), 90)


@pytest.mark.parametrize("physics", ["elastic", "acoustic", "sh", "tmem"])
@pytest.mark.parametrize("rows", [1, 2, 4, 8])
@pytest.mark.parametrize("order,tile,damping,fs", [(2, "least", 2, 0), (8, "least", 1, 0), (8, "odd", 2, 0),
                                                   (8, "most", 2, 1), (12, "most", 2, 0), (4, "odd", 1, 1),
                                                   (12, "odd", 0, 0)])
def test_resident_rows_per_wavefront(physics, rows, order, tile, damping, fs):
    """Every kernel variant, with the smallest block (one halo high), one of an odd number of wavefronts and the
    largest, over tiles that are cut at the right and at the bottom, inside a wavefront's rows too."""
    waves = {"least": max(1, -(-order // 2 // rows)), "odd": 5 if rows < 4 else 3, "most": 16 if rows < 8 else 8}[tile]
    if waves * rows < order // 2:
        waves = 7
    R = waves * rows
    NY = max(3 * order, 2 * R + R // 2 + 3, 45)
    c = _case(physics, 150, NY, 150, order, 2, damping, fs=fs if physics != "tmem" else 0, W=10)
    _equal(c, 150, pieces=[25], plan=(rows, waves))


@pytest.mark.parametrize("physics", ["elastic", "acoustic", "sh", "tmem"])
@pytest.mark.parametrize("order", [2, 4, 6, 8, 10, 12])
def test_resident_plans_fit_the_device(physics, order):
    """The planner counts no more blocks than are resident at once: with shots enough for the whole chip, every
    division of the work runs in the loop, and none is refused at its check-in."""
    c = _case(physics, 70, 45, 16, order, 1, 0)
    c.shots = c.shots * 700
    s = cases.make_solver(c)
    L = wavesim.load()
    wavesim._abi.check(L.wv_set_kernel_timing(s._h, 1))
    for rows in (1, 2, 4, 8):
        for waves in range(1, 17):
            try:
                plan = s.resident_plan(rows, waves)
            except wavesim.WaveError:
                continue
            wavesim._abi.check(L.wv_set_kernel_timing(s._h, 1))
            s.run(0, 16)
            name, n = C.c_char_p(), C.c_longlong()
            wavesim._abi.check(L.wv_kernel_stats(s._h, 0, C.byref(name), None, C.byref(n), None))
            assert name.value == b"res2d" and n.value == 16, plan


@pytest.mark.parametrize("physics", ["elastic", "acoustic"])
@pytest.mark.parametrize("damping", [1, 2])
def test_resident_free_surface(physics, damping):
    _equal(_case(physics, 150, 70, 120, 8, 2, damping, fs=1), 120)


@pytest.mark.parametrize("physics", ["elastic", "tmem"])
def test_resident_run_in_pieces_and_stencil_operators(physics):
    c = _case(physics, 100, 75, 100, 8, 1, 2)
    a = cases.make_solver(c, ops_mode="stencil")
    b = cases.make_solver(c, ops_mode="stencil", path=TWO[physics], tile_y=16)
    for t0, t1 in ((0, 40), (40, 43), (43, 99), (99, 100)):
        a.run(t0, t1)
    b.run(0, 100)
    assert np.array_equal(a.seismograms(0), b.seismograms(0))


def test_resident_many_sources_and_receivers():
    """More than 64 sources in one tile, on shared cells too, and more receivers than a block has threads."""
    c = _case("elastic", 140, 90, 60, 8, 1, 2)
    rng = np.random.default_rng(3)
    sh = c.shots[0]
    cells = np.concatenate([30 + np.arange(70) % 20 + (40 + np.arange(70) // 20) * 140, [30 + 40 * 140] * 5])
    sh.src_index = cells
    sh.src_type = np.array([1 + k % 3 for k in range(len(cells))], np.int32)
    sh.src_signal = rng.standard_normal((len(cells), 60)).astype(np.float32)
    sh.rec_index = np.tile(np.arange(20, 120) + 45 * 140, 25)
    sh.rec_type = np.repeat([1, 2, 3, 2, 1], 500).astype(np.int32)
    _equal(c, 60)


def test_resident_rounds_of_shots():
    """More shots than the chip holds at once: the blocks take them in rounds."""
    _equal(_case("elastic", 300, 200, 200, 8, 23, 2), 200)


@pytest.mark.parametrize("physics", ["elastic", "acoustic", "sh", "tmem"])
@pytest.mark.parametrize("rows,axis,cell", [(0, "x", (20, 100)), (0, "y", (75, 20)), (4, "x", (20, 100)),
                                            (4, "y", (75, 11)), (8, "y", (75, 131))])
def test_resident_infinities_beside_the_frame(physics, rows, axis, cell):
    """A field that overflows: cells that a CPML frame only shares a tile or a wavefront with have no memory
    variables, so an infinite derivative stays one, as in the two-launch kernels (0 times infinity is NaN)."""
    NX, NY, NT = 150, 140, 20
    c = _case(physics, NX, NY, NT, 4, 1, 2, W=9)
    # a field that is differentiated along the axis, and receivers of what its derivative goes to
    field = {"x": {"elastic": 2, "acoustic": 2, "sh": 1, "tmem": 1},
             "y": {"elastic": 4, "acoustic": 2, "sh": 2, "tmem": 0}}[axis][physics]
    sh = c.shots[0]
    xy = [(x, y) for y in range(cell[1] - 6, cell[1] + 7) for x in range(cell[0] - 6, cell[0] + 7)]
    sh.rec_index = np.array([x + y * NX for x, y in xy])
    sh.rec_type = np.full(len(xy), {"sh": 4, "elastic": 2, "tmem": 1, "acoustic": 2 if axis == "x" else 3}[physics],
                          np.int32)
    seis, fields = [], []
    for kw in (dict(), dict(path=TWO[physics], tile_y=16)):
        s = cases.make_solver(c, **kw)
        if rows and not kw:
            s.resident_plan(rows, 8)
        w = s.wavefield(field, 0)
        w[cell[0] + cell[1] * NX] = np.inf
        s.set_wavefield(field, w, 0)
        s.run(0, NT)
        seis.append(s.seismograms(0))
        fields.append([s.wavefield(k, 0) for k in range(5 if physics == "elastic" else 3)])
    assert np.isinf(seis[1]).any()
    assert np.array_equal(seis[0], seis[1], equal_nan=True)
    for a, b in zip(*fields):
        assert np.array_equal(a, b, equal_nan=True)


def test_resident_runs_are_queued():
    """wv_run does not wait for the device: four run calls on each of two handles return while the first is at work
    (0.01 s of a run of about 0.1 s), and both end with the seismograms of handles run one by one."""
    c = _case("elastic", 300, 200, 6000, 8, 2, 2)
    ref = cases.make_solver(c)
    ref.run(0, 6000)
    want = [ref.seismograms(k) for k in range(2)]
    hs = [cases.make_solver(c) for _ in range(2)]
    for h in hs:
        h.run(0, 6000)
        h.synchronize()
        h.reset()
    t0 = time.perf_counter()
    for n in range(4):
        for h in hs:
            h.run(1500 * n, 1500 * n + (1500 if n < 3 else 1495))
    for h in hs:
        h.run(5995, 6000)
    queued = time.perf_counter() - t0
    for h in hs:
        h.synchronize()
    total = time.perf_counter() - t0
    assert queued < total / 4, (queued, total)
    for h in hs:
        for k in range(2):
            assert np.array_equal(h.seismograms(k), want[k])


def test_resident_record_gives_the_same_gradient():
    """The record of the derivative sums written by the resident loop (rows per wavefront as the strips of
    the record) leads to the gradient of the row-strip kernels' record."""
    c = cases.elastic_c4(N=130, NT=120, nshots=3, W=10)
    g = []
    for ty in (16, 0):
        sol = cases.make_solver(c, path="strip", tile_y=ty)
        sol.set_checkpointing(40, True)
        sol.run(0, 120)
        for k in range(3):
            sol.set_adjoint_source(k, sol.seismograms(k))
        sol.run_adjoint()
        g.append([sol.gradient(p) for p in ("vp", "vs", "rho")])
    for x, y in zip(*g):
        # (the adjoint pass adds its FP64 terms with atomics, in no fixed order)
        assert np.linalg.norm(x - y) <= 1e-12 * np.linalg.norm(y)
