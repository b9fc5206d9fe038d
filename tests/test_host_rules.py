"""Rules by which the host chooses kernels, on the CPU.

* The classes of the batched line kernels (chunk length, threads per row):
  every class that the shape rule or a tuning table can choose has a kernel in
  the launch of several classes, and the host knows the others from these (a
  workgroup of an unknown class would do nothing).
* The red-black tile of a level that is not timed: the small one below 256^2
  cells, the one with the fewest window cells for larger levels (a level met
  while its stream is being captured)."""
import ctypes

import pytest

mg = pytest.importorskip("mgpoisson2d_amd.capi")

KERNELS = {(2, 64), (4, 64), (8, 64), (2, 128), (4, 128), (8, 128), (2, 256), (4, 256), (8, 256), (16, 256)}


def native(name, *argtypes, res=ctypes.c_int):
    f = getattr(mg.lib, name)
    f.restype, f.argtypes = res, argtypes
    return f


def test_known_classes():
    known = native("_ZN3mgp17xline_batch_classEii", ctypes.c_int, ctypes.c_int, res=ctypes.c_bool)
    got = {(C, t) for C in range(1, 65) for t in (32, 64, 128, 256, 512, 1024) if known(C, t)}
    assert got == KERNELS


def test_chosen_classes_are_known():
    shape = native("_ZN3mgp17xline_batch_shapeEiRiS0_", ctypes.c_int, ctypes.POINTER(ctypes.c_int),
                   ctypes.POINTER(ctypes.c_int), res=None)
    chunk = native("_ZN3mgp17xline_batch_chunkEiim", ctypes.c_int, ctypes.c_int, ctypes.c_size_t)
    for nx in range(4, 4112):
        C, t = ctypes.c_int(), ctypes.c_int()
        shape(nx, ctypes.byref(C), ctypes.byref(t))
        assert (C.value, t.value) in KERNELS, nx
        for width in (64, 128, 256):
            for elem in (4, 8):
                c = chunk(nx, width, elem)
                assert c == 0 or (c, width) in KERNELS, (nx, width, elem)


def test_untimed_red_black_tile():
    untimed = native("_ZN3mgp18dc_rb_tile_untimedEiii", ctypes.c_int, ctypes.c_int, ctypes.c_int)
    shapes = [(16, 4), (32, 4), (32, 8), (64, 8), (16, 8)]  # window rows, waves
    width = 128  # window columns

    def cells(nx, ny, S, k):
        tx, ty = width - 4 * S, shapes[k][0] - 4 * S
        return -(-nx // tx) * -(-ny // ty) * width * shapes[k][0]

    for S in (1, 2):
        for nx, ny in [(8, 8), (64, 64), (255, 256)]:
            assert shapes[untimed(nx, ny, S)] == (16, 8)
        for nx, ny in [(256, 256), (300, 700), (2048, 2048), (2500, 40)]:
            k = untimed(nx, ny, S)
            assert cells(nx, ny, S, k) == min(cells(nx, ny, S, q) for q in range(len(shapes))), (nx, ny, S, k)
