"""Calls of several steps (psl_update_grid) against the same steps one call at a
time: the periodic copies passed on inside the update, and the box-face cells
updated in the bulk kernel or staged, leave the same bits in every cell."""
import ctypes
import threading

import numpy as np
import pytest

from periodicshiftlbm_amd import cases

pytestmark = pytest.mark.gpu


def _grid(P, shape, storage, copies, seed, flags=None):
    rng = np.random.default_rng(seed)
    nx, ny, nz = shape
    n = nx * ny * nz
    g = P.GridStruct(P.InfoStruct(cellCountX=nx, cellCountY=ny, cellCountZ=nz, nu=0.01), storage)
    if flags is not None:
        g.set_flags(flags)
        g.set_given_values(cases.channel_given_values(0.03))
    g.set_smagorinsky(0.12 if seed % 2 else 0.0)
    g.set_periodic_copies(x=copies[0], y=copies[1])
    P.fill_equilibrium(g, rng.uniform(0.98, 1.02, n).astype(np.float32),
                       *rng.uniform(-0.03, 0.03, (3, n)).astype(np.float32))
    return g


def _same(a, b, what):
    assert a.shifter.tolist() == b.shifter.tolist()
    nbad = int(np.count_nonzero(a.get_f().view(np.uint32) != b.get_f().view(np.uint32)))
    assert nbad == 0, f"{what}: {nbad} values differ"


# (from 32768 cells on, FP32; 16-bit grids from 45000 or 70000 on) rows shorter than, equal to and longer than a wave and a
# workgroup; single and double layers on every axis, where a copied face is its
# own or its neighbour's
SHAPES = [(2, 130, 128), (3, 200, 60), (5, 100, 70), (17, 50, 41), (63, 3, 180), (64, 4, 130), (65, 5, 110),
          (130, 2, 130), (257, 9, 15), (300, 1, 112), (2, 1, 20000), (17000, 2, 1), (40000, 1, 1)]
SHAPES_16BIT = [(2, 300, 140), (3, 300, 100), (5, 150, 120), (17, 70, 70), (63, 5, 270), (64, 4, 330), (65, 5, 260),
                (130, 2, 330), (257, 18, 19), (300, 1, 280), (2, 1, 45000), (45000, 2, 1), (90000, 1, 1)]


@pytest.mark.parametrize("storage", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("copies", [(True, False), (True, True)])
def test_copies_inside_a_call_equal_copy_passes(psl, storage, copies):
    P = psl
    for s, shape in enumerate(SHAPES + (SHAPES_16BIT if storage != "f32" else [])):
        n = shape[0] * shape[1] * shape[2]
        solid = None
        if s % 3 == 2:  # bounceback cells, on the copied faces too
            solid = np.where(np.random.default_rng(s).random(n) < 0.2, cases.BOUNCEBACK, cases.FLUID).astype(np.uint8)
        a, b = (_grid(P, shape, storage, copies, s, solid) for _ in range(2))
        for steps in (2, 5):
            P.updateGrid([a], steps)
            for _ in range(steps):
                P.updateGrid([b], 1)
            _same(a, b, f"{shape} after {steps}")
        a.close()
        b.close()


@pytest.mark.parametrize("storage,shape", [("f32", (65, 41, 40)), ("f16", (65, 36, 35)), ("bf16", (63, 37, 36))])
@pytest.mark.parametrize("solid", [False, True])
def test_copies_inside_a_call_at_every_variant(psl, storage, shape, solid):
    """The non-temporal forms of the update with copies through the ring."""
    P = psl
    n = shape[0] * shape[1] * shape[2]
    flags = None
    if solid:
        flags = np.where(np.random.default_rng(3).random(n) < 0.2, cases.BOUNCEBACK, cases.FLUID).astype(np.uint8)
    b = _grid(P, shape, storage, (True, True), 1, flags)
    for _ in range(4):
        P.updateGrid([b], 1)
    for v in range(P.TUNE_VARIANTS):
        a = _grid(P, shape, storage, (True, True), 1, flags)
        a.tuning = v
        P.updateGrid([a], 4)
        _same(a, b, f"{storage} {shape} variant {v}")
        a.close()
    b.close()


def test_no_ring_memory_where_the_copies_stay_passes(psl):
    """A ring of 64 MB for the x copies is made by the first call that uses it, not
    for a grid with listed cells, whose copies stay passes."""
    P = psl

    def free():
        P.synchronize()
        f, total = ctypes.c_size_t(0), ctypes.c_size_t(0)
        assert P.lib().hipMemGetInfo(ctypes.byref(f), ctypes.byref(total)) == 0  # of the runtime psl is linked to
        return f.value

    shape = (4, 512, 512)
    n = shape[0] * shape[1] * shape[2]
    flags = np.zeros(n, np.uint8)
    flags[: shape[0] * shape[1]] = cases.GIVEN_U | cases.PERIODIC_X | cases.PERIODIC_Y  # listed z face
    for listed in (True, False):
        g = _grid(P, shape, "f32", (True, False), 1, flags if listed else None)
        P.updateGrid([g], 1)
        before = free()
        P.updateGrid([g], 2)
        used = before - free()
        print(f"  listed {listed}: {used / 2**20:.1f} MB more", flush=True)
        assert used < 16 << 20 if listed else used >= 64 << 20
        g.close()


@pytest.mark.parametrize("mode", [0, 1, 2])  # global, thread-local, relaxed
def test_first_ring_call_leaves_another_threads_capture_valid(psl, mode):
    """The rings are allocated inside the first call of several steps; a capture that
    another thread has begun on a stream of its own still ends well, and so does
    the call."""
    P = psl
    hip = P.lib()  # symbols of the runtime psl is linked to
    streams = [ctypes.c_void_p() for _ in range(2)]
    for s in streams:
        assert hip.hipStreamCreateWithFlags(ctypes.byref(s), 1) == 0
    a, b = (_grid(P, (65, 41, 40), "f32", (True, True), 1) for _ in range(2))
    for g in (a, b):
        P.synchronize()
        g.set_stream(streams[0].value)
        P.updateGrid([g], 1)
    P.synchronize()
    begun, stepped, rc = threading.Event(), threading.Event(), []

    def capture():
        graph = ctypes.c_void_p()
        rc.append(hip.hipStreamBeginCapture(streams[1], mode))
        begun.set()
        stepped.wait(60)
        rc.append(hip.hipStreamEndCapture(streams[1], ctypes.byref(graph)))
        if graph:
            hip.hipGraphDestroy(graph)

    t = threading.Thread(target=capture)
    t.start()
    begun.wait(60)
    try:
        P.updateGrid([a], 4)
    finally:
        stepped.set()
        t.join()
    P.synchronize()
    assert rc == [0, 0]
    for _ in range(4):
        P.updateGrid([b], 1)
    P.synchronize()
    _same(a, b, f"capture mode {mode}")
    for g in (a, b):
        g.close()
    for s in streams:
        hip.hipStreamDestroy(s)


# FP16 / BF16 grids of 66 MB are staged, and FP16 ones of 274 MB; 20 MB, BF16 of 307 MB, FP16 of
# 356 MB, and every FP32 grid, are updated in place
@pytest.mark.parametrize("storage,shape", [("f16", (128, 100, 100)), ("bf16", (130, 99, 101)), ("f16", (74, 73, 72)),
                                           ("f16", (260, 145, 141)), ("f32", (131, 70, 69)), ("f16", (300, 151, 153)),
                                           ("bf16", (287, 145, 143))])
def test_box_faces_staged_and_in_place_equal_the_fused_launch(psl, storage, shape):
    P = psl
    rng = np.random.default_rng(3)
    flags = cases.channel_flags(shape, rng.random(shape[0] * shape[1] * shape[2]) < 0.02)
    a, b = (_grid(P, shape, storage, (False, True), 3, flags) for _ in range(2))
    b.tuning = P.TUNE_FUSED_BOUNDARY
    P.updateGrid([a], 3)
    P.updateGrid([b], 3)
    _same(a, b, f"{storage} {shape}")
    a.close()
    b.close()
