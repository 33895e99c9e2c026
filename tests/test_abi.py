"""The C-ABI library loads and exports every entry point include/wave_abi.h declares (no GPU needed)."""
import ctypes
import os
import re

import wavesim._abi as abi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared():
    text = open(os.path.join(ROOT, "include", "wave_abi.h")).read()
    return sorted(set(re.findall(r"^\s*(?:int|const char \*)\s*(wv_\w+)\s*\(", text, re.M)))


def test_header_matches_binding_list():
    assert _declared() == sorted(abi.EXPORTS)


def test_library_exports_every_symbol():
    lib = ctypes.CDLL(abi.LIB_PATH)
    for name in _declared():
        assert hasattr(lib, name), name


def test_last_error_is_callable_without_gpu():
    lib = abi.load()
    assert isinstance(lib.wv_last_error(), bytes)


def test_factory_rejects_unknown_types_without_gpu():
    """ForwardSolverFactory.cpp:4-66 throws on unknown dimension/type; the ABI returns WV_EINVAL."""
    lib = abi.load()
    h = ctypes.c_void_p()
    assert lib.wv_create(b"4D", b"elastic", ctypes.byref(h)) == -1
    assert b"dimension" in lib.wv_last_error()
    assert lib.wv_create(b"2D", b"plasma", ctypes.byref(h)) == -1
    # factory types this build does not provide
    # (the reference factory returns an empty pointer for 3D tmem / sh / viscosh / viscotmem)
    for d, t in ((b"3D", b"tmem"), (b"3D", b"sh"), (b"3D", b"viscosh"), (b"3D", b"viscotmem")):
        assert lib.wv_create(d, t, ctypes.byref(h)) == -1, (d, t)
        assert b"not provided" in lib.wv_last_error()
    # and the ones it does (creation touches no GPU)
    for d, t in ((b"2D", b"viscoelastic"), (b"2D", b"viscosh"), (b"2D", b"sh"), (b"2D", b"emem"), (b"3D", b"acoustic"),
                 (b"3D", b"viscoelastic"), (b"2D", b"viscotmem"), (b"2D", b"viscoemem")):
        assert lib.wv_create(d, t, ctypes.byref(h)) == 0, (d, t)
        lib.wv_destroy(h)


def test_depth_parts_are_never_empty():
    """The 3D kernels' parts along depth (wv::depth_parts): every part holds planes, and the rule's
    bounds (at least max(4H, 8) planes wanted per part, no more parts than the block count asks for) hold."""
    f = ctypes.CDLL(abi.LIB_PATH)["_ZN2wv11depth_partsEiiii"]
    f.argtypes, f.restype = [ctypes.c_int] * 4, ctypes.c_int
    for H in range(1, 7):
        for tiles in (1, 7, 96, 480, 1500, 20000):
            for NY in range(2, 420):
                n = f(NY, H, tiles, 12288)
                wanted = max(1, min(-(-12288 // tiles), NY // max(4 * H, 8)))
                assert 1 <= n <= wanted
                planes = -(-NY // n)
                assert (n - 1) * planes < NY <= n * planes, (NY, H, tiles, n)
                assert planes == -(-NY // wanted)


def test_depth_parts_fill_the_chip():
    """wv::depth_parts_fill: the parts of depth_parts, or more of at least 2 planes, none empty, where
    those leave part of the chip's block slots free; then no more blocks than slots."""
    lib = ctypes.CDLL(abi.LIB_PATH)
    f, g = lib["_ZN2wv11depth_partsEiiii"], lib["_ZN2wv16depth_parts_fillEiiiii"]
    f.argtypes, f.restype = [ctypes.c_int] * 4, ctypes.c_int
    g.argtypes, g.restype = [ctypes.c_int] * 5, ctypes.c_int
    for H in range(1, 7):
        for tiles in (1, 7, 40, 96, 480, 1500, 20000):
            for slots in (256, 512, 1280):
                for NY in range(2, 300):
                    n, m = f(NY, H, tiles, 12288), g(NY, H, tiles, 12288, slots)
                    planes = -(-NY // m)
                    assert (m - 1) * planes < NY <= m * planes, (NY, H, tiles, slots, m)
                    if m > n:
                        assert m * tiles <= slots and planes >= 2
                    elif m < n:
                        raise AssertionError((NY, H, tiles, slots))
                    elif n * tiles < slots:  # nothing more fits: one plane less per part is too many blocks
                        p = -(-NY // n) - 1
                        assert p < 2 or -(-NY // p) * tiles > slots
